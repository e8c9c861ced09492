"""The projection GEMM in every tile size, through the C ABI: grids whose cell count 256 (or
128) does not divide, the smallest ones and every head width, against an fp64 product.

Bound per element, from the data types: fp32 sums of K products in any order are off by at
most (K + 2) u sum |x||w|, u = 2^-24; the activations change a value by at most a factor
1.13 (GELU's slope) plus 1e-6 (|v| + 1) for exp2 and the reciprocal; bf16 storage rounds
each output by at most half a unit of its 8-bit significand, 2^-8 |v|. Chained planes carry the previous plane's error through |W|, so
they are checked plane by plane on the device's own input plane.
"""
import numpy as np
import pytest

from slime_amd import Pseudopod, round_bf16

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(autouse=True)
def _needs_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


def _gelu(v):
    return 0.5 * v * (1 + torch.tanh(0.7978845608028654 * (v + 0.044715 * v ** 3)))


def _check(got, x, w, act, bf16, name):
    """got [n, C] against act(x w): x [n, K], w [K, C] on the device."""
    x, w = x.double(), w.double()
    v = x @ w
    bound = (x.shape[1] + 2) * 2.0 ** -24 * (x.abs() @ w.abs())
    ref = torch.relu(v) if act == 1 else _gelu(v) if act == 2 else v
    bound = 1.13 * bound + 1e-6 * (v.abs() + 1) * (act == 2)
    if bf16:
        bound = bound * 1.01 + 2.0 ** -8 * ref.abs()
    over = (got.double() - ref).abs() - bound
    assert torch.isfinite(got.float()).all(), name
    assert float(over.max()) <= 0.0, (name, float(over.max()))


@pytest.mark.parametrize("dtype", ["bf16", "fp32"])
@pytest.mark.parametrize("B,G,D,pods,chain", [
    # The rows of a pod are one batch of the product; test_gemm_rule.py holds the tiles.
    (1, 8, 8, 1, 0),      # one 64-row tile, the narrowest heads
    (3, 8, 64, 3, 0),     # a pod per tile of rows
    (2, 24, 16, 1, 0),    # 1152 rows over two batch entries in 64-wide tiles
    (4, 40, 32, 2, 1),
    (2, 56, 64, 2, 0),    # 3136 rows per pod: bf16 in 128-wide tiles, the last one moved back by half
    (1, 72, 8, 1, 2),
    (1, 88, 64, 1, 0),    # 7744 rows in 128-wide tiles, the last one moved back by half
    (6, 136, 64, 2, 0),   # 55,488 rows per pod, likewise
    (4, 136, 64, 1, 0),   # 73,984 rows: 256-wide tiles, which one batch entry's 18,496 do not fill
])
def test_projections_match_fp64(dtype, B, G, D, pods, chain):
    print(f"[case] {dtype} B={B} G={G} D={D} pods={pods} chain={chain}", flush=True)
    C, bf16 = 8 * D, dtype == "bf16"
    rng = np.random.default_rng(G + D)
    p = {k: rng.normal(0, 0.1, (pods, C, C)).astype(np.float32) for k in ("WP", "WI", "WV")}
    if bf16:
        p = {k: round_bf16(v) for k, v in p.items()}
    p.update(K=rng.normal(0, 0.05, (pods, 8, 9)), M=np.tile(np.eye(8), (pods, 1, 1)),
             mu=np.full((pods, 8), 0.2), sigma=np.full((pods, 8), 0.05))
    g = torch.Generator(device="cuda").manual_seed(G)
    x = torch.randn(B, G, G, C, generator=g, device="cuda").to(torch.bfloat16 if bf16 else torch.float32)
    with Pseudopod(B, G, 8, D, dtype, pods=pods, pvi_chain=chain) as e:
        e.set_params(p)
        P, I, V = e.project(x)
        torch.cuda.synchronize()
    xs = x
    if chain == 2:  # the 3x3 neighbourhood sum, rounded to the storage type as the library keeps it
        xs = sum(x.float().roll((dy, dx), (1, 2)) for dy in (1, 0, -1) for dx in (1, 0, -1)).to(x.dtype)
    for b in range(B):
        w = [torch.from_numpy(p[k][b // (B // pods)]).cuda() for k in ("WP", "WI", "WV")]
        ins = [xs[b], P[b] if chain else x[b], I[b] if chain else x[b]]
        for got, src, wk, act, name in zip((P, I, V), ins, w, (1, 2, 0), "PIV"):
            _check(got[b].reshape(G * G, C), src.reshape(G * G, C), wk, act, bf16, (name, b))


@pytest.mark.parametrize("dtype,G,D", [("fp32", 24, 16), ("bf16", 40, 64), ("fp32", 16, 64)])
def test_project_takes_a_state_inside_another_buffer(dtype, G, D):
    """A contiguous state that starts one element into its buffer, which no 16-byte load fits."""
    C, bf16 = 8 * D, dtype == "bf16"
    rng = np.random.default_rng(D)
    p = {k: rng.normal(0, 0.1, (1, C, C)).astype(np.float32) for k in ("WP", "WI", "WV")}
    if bf16:
        p = {k: round_bf16(v) for k, v in p.items()}
    p.update(K=np.zeros((1, 8, 9)), M=np.eye(8)[None], mu=np.full((1, 8), 0.2), sigma=np.full((1, 8), 0.05))
    dt = torch.bfloat16 if bf16 else torch.float32
    buf = torch.randn(1 + G * G * C, generator=torch.Generator(device="cuda").manual_seed(1), device="cuda").to(dt)
    x = buf[1:].view(1, G, G, C)
    assert x.is_contiguous() and x.data_ptr() % 16
    with Pseudopod(1, G, 8, D, dtype) as e:
        e.set_params(p)
        outs = e.project(x)
        torch.cuda.synchronize()
    for got, k, act in zip(outs, ("WP", "WI", "WV"), (1, 2, 0)):
        _check(got.reshape(G * G, C), x.reshape(G * G, C), torch.from_numpy(p[k][0]).cuda(), act, bf16, k)

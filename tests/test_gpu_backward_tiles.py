"""The backward's products at shapes off the 256-wide tiles -- ragged grids (576 and 1600 rows
per pod: row chunks with a remainder), C = 64 in bf16 and every fp32 width, and the taped
projections and dX in 128-wide tiles, the last one moved back to the pod's end
(test_gemm_rule.py holds which tiles these are) -- against the oracle's fp64 gradient, with the bounds of
test_gpu_backward (normalised maximum 1e-5 for an fp32 state, 2e-2 for bf16)."""
import pytest

from tests.conftest import norm_err
from tests.test_gpu_backward import NAMES, TOL, _cfg, _dev, _inputs

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from slime_amd import Pseudopod  # noqa: E402


@pytest.mark.parametrize("dtype,D,pods,B,G", [
    ("bf16", 8, 2, 4, 24),
    ("bf16", 16, 1, 1, 40),
    ("bf16", 64, 1, 1, 24),
    ("fp32", 8, 1, 1, 40),
    ("fp32", 32, 2, 2, 24),
    ("fp32", 64, 1, 2, 24),
    # 128-wide tiles: 3136 and 7744 rows per pod (the last tile moved back by half), 8192 rows
    ("bf16", 64, 2, 2, 56),
    ("fp32", 64, 1, 1, 88),
    ("fp32", 64, 1, 2, 64),
])
def test_backward_products_match_oracle(oracle, dtype, D, pods, B, G):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    print(f"[case] backward {dtype} D={D} pods={pods} B={B} G={G}", flush=True)
    cfg = _cfg(B=B, G=G, D=D, dtype=dtype, pods=pods)
    p, X, T = _inputs(cfg)
    with Pseudopod(B, G, 8, D, dtype, cfg.dt, False, pods) as e:
        e.set_params(p)
        loss, gx, grads = e.backward(_dev(X, dtype), _dev(T, dtype))
        torch.cuda.synchronize()
        gx = gx.cpu().numpy()
        grads = {k: v.cpu().numpy() for k, v in grads.items()}
    rloss, ref = oracle.step_backward(oracle.OracleConfig(B=B, G=G, H=8, D=D, pods=pods), X, p, T)
    assert abs(loss - rloss) <= TOL[dtype] * rloss
    errs = {"X": norm_err(gx, ref["X"]), **{k: norm_err(grads[k], ref[k]) for k in NAMES}}
    print("  normalised errors " + " ".join(f"{k}={v:.2e}" for k, v in errs.items()))
    for k, v in errs.items():
        assert v <= TOL[dtype], (k, v)

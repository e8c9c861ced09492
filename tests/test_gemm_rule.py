"""The tile that each projection GEMM of the GPU tests runs in, by the library's own rule
(``slime_amd/csrc/gemm_rule.hpp``) on the MI355X's 256 CUs: which kernel a case covers."""
import itertools
import random

import pytest

from tests.gemm_launches import build_rule_query, launches, tiles

FIRST, LATER, DX = 0, 1, 6  # indices into launches()


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    return build_rule_query(tmp_path_factory.mktemp("rule"))


def _cases(test):
    """The parametrised values of a test, as dicts (the marks' lists, multiplied out)."""
    lists = []
    for m in test.pytestmark:
        if m.name == "parametrize":
            keys = m.args[0].split(",")
            lists.append([dict(zip(keys, v if len(keys) > 1 else (v,))) for v in m.args[1]])
    for combo in itertools.product(*lists):
        yield {k: v for d in combo for k, v in d.items()}


def test_projection_cases_cover_every_tile(rule):
    from tests import test_gpu_gemm_tiles as t
    want = {(1, 8, 8): 64, (3, 8, 64): 64, (2, 24, 16): 64, (4, 40, 32): 64, (1, 72, 8): 64, (1, 88, 64): 128,
            (6, 136, 64): 128, (4, 136, 64): 256}
    for c in _cases(t.test_projections_match_fp64):
        first = launches(c["B"], c["G"], c["D"], c["dtype"], c["pods"])[FIRST]
        got = tiles(rule, [first])[0]
        expect = want.get((c["B"], c["G"], c["D"]), 128 if c["dtype"] == "bf16" else 64)  # (2, 56, 64)
        if c["chain"] == 0:
            assert got == expect, (c, got)


def test_backward_cases_cover_the_tape_and_the_addend_in_every_tile(rule):
    """(dtype, tile) of the taped projections and of dX over test_gpu_backward_tiles.py."""
    from tests import test_gpu_backward_tiles as t
    tape, dx = set(), set()
    for c in _cases(t.test_backward_products_match_oracle):
        L = launches(c["B"], c["G"], c["D"], c["dtype"], c["pods"])
        got = tiles(rule, [L[FIRST], L[DX]])
        tape.add((c["dtype"], got[0]))
        dx.add((c["dtype"], got[1]))
    small = {(d, t_) for d in ("bf16", "fp32") for t_ in (64, 128)}
    assert tape >= small and dx >= small, (tape, dx)


def test_large_configurations_take_the_256_wide_tile(rule):
    from slime_amd.synthetic import CONFIGS
    for name in ("c3", "c4", "c5"):
        c = CONFIGS[name]
        L = launches(c.B, c.G, c.D, c.dtype, c.pods)
        assert tiles(rule, [L[FIRST], L[LATER], L[DX]]) == [256, 256, 256], name


def test_every_accepted_configuration_has_a_tile(rule):
    """slime_ca_uses_mfma is 1 for every handle: some tile fits every launch of every shape that
    slime_ca_create takes (G a multiple of 8, D of 8, 16, 32, 64, pods dividing B)."""
    rng = random.Random(1)
    todo = []
    for D, dtype in itertools.product((8, 16, 32, 64), ("bf16", "fp32")):
        for G in list(range(8, 129, 8)) + [512]:
            B = rng.choice((1, 2, 3, 6))
            pods = rng.choice([p for p in range(1, B + 1) if B % p == 0])
            todo += launches(B, G, D, dtype, pods)
    for n_cu in (256, 80):
        assert 0 not in tiles(rule, todo, n_cu)

"""Host replay of the 128- and 64-wide tile GEMM's addresses and waits (CPU only): every direct
load, LDS slot and fragment read of a launch, and the three-stage ring's waits, through
the kernel's own functions (``slime_amd/csrc/gemm_small_addr.hpp``), at ragged grids, the
smallest ones and every head width; the launches are the library's
(``tests/gemm_launches.py``)."""
import os
import subprocess

import pytest

from tests.gemm_launches import launches

SRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "gemm_small_replay.cpp")


@pytest.fixture(scope="module")
def replay(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("replay") / "gemm_small_replay")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", "-o", exe, SRC], check=True)
    return exe


def _run(exe, tile, L, extra=()):
    args = [tile, 64 if tile == 128 else 128, L.M, L.N, L.K, L.elem, L.rows_per_batch, L.bt_batch_stride,
            L.bt_elems, L.ncol]
    r = subprocess.run([exe, *map(str, args), *extra], capture_output=True, text=True, timeout=120)
    return r.returncode, r.stdout.strip()


@pytest.mark.parametrize("dtype", ["bf16", "fp32"])
@pytest.mark.parametrize("tile,B,G,D,pods", [
    (64, 1, 8, 8, 1),      # one tile of rows, the narrowest heads
    (64, 3, 8, 64, 3),
    (64, 2, 24, 32, 1),
    (64, 4, 40, 32, 2),
    (128, 2, 16, 16, 1),
    (128, 3, 24, 64, 3),   # 576 rows per batch: a last tile moved back by half
    (128, 3, 24, 64, 1),   # 1728 over the pod: likewise
    (128, 1, 40, 16, 1),
    (128, 2, 32, 32, 2),
    (128, 6, 136, 64, 2),
])
def test_every_address_of_a_launch(replay, tile, B, G, D, pods, dtype):
    for L in launches(B, G, D, dtype, pods):
        rc, out = _run(replay, tile, L)
        assert rc == 0, (L.name, out)


def test_a_tile_past_the_batch_is_reported(replay):
    rc, out = _run(replay, 128, launches(3, 24, 64, "bf16")[1], ["past-end"])
    assert rc == 1 and "outside its batch" in out, out


def test_a_loose_wait_is_reported(replay):
    rc, out = _run(replay, 128, launches(3, 24, 64, "bf16")[0], ["loose-wait"])
    assert rc == 1 and "too loose" in out, out


def test_weights_of_a_pod_read_per_batch_entry_are_reported(replay):
    first, later = launches(3, 24, 64, "bf16")[:2]
    rc, out = _run(replay, 128, later._replace(bt_elems=first.bt_elems))
    assert rc == 1 and "direct load out of range" in out, out

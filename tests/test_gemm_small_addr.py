"""Host replay of the 128- and 64-wide tile GEMM's addresses (CPU only): every direct load,
LDS slot and fragment read of a launch through the kernel's own address functions
(``slime_amd/csrc/gemm_small_addr.hpp``), at ragged grids, the smallest ones and every
head width; the launches are the library's forward and dX products."""
import os
import subprocess

import pytest

SRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "gemm_small_replay.cpp")


@pytest.fixture(scope="module")
def replay(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("replay") / "gemm_small_replay")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", "-o", exe, SRC], check=True)
    return exe


def _run(exe, tile, B, G, D, elem, kind, extra=()):
    C, rpb = 8 * D, G * G
    N, K = (3 * C, C) if kind == "forward" else (C, 3 * C)
    args = [tile, 64 if tile == 128 else 128, B * rpb, N, K, elem, rpb, 3 * C * C, B * 3 * C * C, C]
    r = subprocess.run([exe, *map(str, args), *extra], capture_output=True, text=True, timeout=120)
    return r.returncode, r.stdout.strip()


@pytest.mark.parametrize("elem", [2, 4])
@pytest.mark.parametrize("kind", ["forward", "dX"])
@pytest.mark.parametrize("tile,B,G,D", [
    (64, 1, 8, 8),      # one tile of rows, the narrowest heads
    (64, 3, 8, 64),
    (64, 2, 24, 32),
    (128, 2, 16, 16),
    (128, 3, 24, 64),   # 576 rows per batch: a last tile moved back by half
    (128, 1, 40, 16),
    (128, 2, 32, 32),
])
def test_every_address_of_a_launch(replay, tile, B, G, D, elem, kind):
    rc, out = _run(replay, tile, B, G, D, elem, kind)
    assert rc == 0, out


def test_a_tile_past_the_batch_is_reported(replay):
    rc, out = _run(replay, 128, 3, 24, 64, 2, "forward", ["past-end"])
    assert rc == 1 and "outside its batch" in out

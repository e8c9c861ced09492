"""The wave-front Jacobi schedule on the CPU: an emulation of fitness_finalize_kernel's lanes
and work items (``slime_amd/csrc/jacobi_wave.hpp``) against the cyclic row order done one
rotation at a time. Both take the same rotations of the same values up to the fp64
rounding of commuted updates (a few units of 2^-53 per rotation chain of 2 D steps and
sweep), so sweep counts agree exactly and diagonals to 1e-12 of the largest."""
import os
import subprocess

import pytest

SRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "jacobi_wave_check.cpp")


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("jacobi") / "jacobi_wave_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", "-o", exe, SRC], check=True)
    return exe


@pytest.mark.parametrize("D", [8, 16, 32, 64])
@pytest.mark.parametrize("kind", ["dense", "lowrank", "diag", "rank1"])
def test_wave_front_is_the_cyclic_order(check, D, kind):
    for seed in (1, 2, 3):
        r = subprocess.run([check, str(D), str(seed), kind], capture_output=True, text=True, timeout=60)
        assert r.returncode == 0, r.stdout


def test_a_stale_element_is_reported(check):
    r = subprocess.run([check, "64", "1", "dense", "swap-order"], capture_output=True, text=True, timeout=60)
    assert r.returncode == 1 and "FAIL" in r.stdout


def test_rotation_is_the_exact_one_to_a_few_roundings(check):
    """Bounds derived from the form's roundings (jacobi_wave.hpp): c 2.3, s 8.3 units of 2^-53."""
    for seed in ("1", "2"):
        r = subprocess.run([check, "rotation", "600000", seed], capture_output=True, text=True, timeout=60)
        print(r.stdout.strip())
        assert r.returncode == 0, r.stdout


@pytest.mark.parametrize("plant", ["sign", "half"])
def test_a_wrong_rotation_is_reported(check, plant):
    r = subprocess.run([check, "rotation", "1000", "1", plant], capture_output=True, text=True, timeout=60)
    assert r.returncode == 1 and "FAIL rotation" in r.stdout

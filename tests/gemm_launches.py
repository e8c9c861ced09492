"""The projection GEMMs that the library launches for a configuration (run_project and
slime_ca_backward, slime_amd/csrc/api.cpp), and the tile its rule picks for each
(slime_amd/csrc/gemm_rule.hpp, through a small g++ build)."""
import os
import subprocess
from collections import namedtuple

HERE = os.path.dirname(os.path.abspath(__file__))

# rows_per_batch: rows of A that share one Bt; bt_elems: elements from Bt to its buffer's end.
Launch = namedtuple("Launch", "name M N K elem rows_per_batch bt_batch_stride bt_elems ncol nplanes epilogue")


def launches(B, G, D, dtype, pods=1):
    """Weights that no mass factor scales are laid out once per pod ([pods][3C][C]): those of a
    call's first step, of project and of the backward's tape, and planes 1 and 2 of a chain.
    Later steps of a call read per-batch ones ([B][3C][C]); dX reads [pods][C][3C]."""
    C, elem = 8 * D, (2 if dtype == "bf16" else 4)
    M, cells, pod_rows = B * G * G, G * G, B // pods * G * G
    stride, per_pod, per_batch = 3 * C * C, pods * 3 * C * C, B * 3 * C * C
    epi = "bf16" if dtype == "bf16" else "f32"
    return [
        Launch("first step [P|I|V]", M, 3 * C, C, elem, pod_rows, stride, per_pod, C, 3, epi),
        Launch("later step [P|I|V]", M, 3 * C, C, elem, cells, stride, per_batch, C, 3, epi),
        Launch("chained plane 0, first step", M, C, C, elem, pod_rows, stride, per_pod, C, 1, epi),
        Launch("chained plane 0, later step", M, C, C, elem, cells, stride, per_batch, C, 1, epi),
        Launch("chained plane 1", M, C, C, elem, pod_rows, stride, per_pod - C * C, C, 1, epi),
        Launch("chained plane 2", M, C, C, elem, pod_rows, stride, per_pod - 2 * C * C, C, 1, epi),
        Launch("backward dX", M, C, 3 * C, elem, pod_rows, stride, per_pod, C, 1, "f32add"),
    ]


def build_rule_query(directory):
    exe = os.path.join(str(directory), "gemm_rule_query")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", "-o", exe,
                    os.path.join(HERE, "gemm_rule_query.cpp")], check=True)
    return exe


def tiles(exe, launches, n_cu=256):
    args = [str(v) for L in launches for v in (int(L.elem == 2), L.M, L.N, L.K, L.ncol, L.rows_per_batch)]
    r = subprocess.run([exe, str(n_cu), *args], capture_output=True, text=True, check=True, timeout=60)
    return [int(v) for v in r.stdout.split()]

"""bench.py on the CPU: its work models against the kernels they describe."""
import math
import os
import re
import sys
import types

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
import bench  # noqa: E402

CSRC = os.path.join(ROOT, "ptychotomo_amd", "csrc")


def _source():
    return "".join(open(os.path.join(CSRC, f)).read() for f in ("tomo.hip", "ptycho.hip"))


def test_probed_kernels_exist():
    """Every probed tag is one that a launch records."""
    tags = set(re.findall(r'ProfScope \w+\((?:[^;"]*\? )?"(\w+)"', _source()))
    assert set(bench.TAGS) <= tags, set(bench.TAGS) - tags


def test_gather_taps_are_the_kernels():
    kw = int(re.search(r"constexpr int kW = (\d+);", _source()).group(1))
    assert bench.GATHER_TAPS == kw * kw


def test_kernel_bytes_of_the_grids():
    """The forward grids 2N x 2N points (N = 3n/2), the adjoint 2n x 2n, both
    within the samples' disc; each kernel's output is the next one's input."""
    n, nz, nt = 64, 10, 96
    slv = types.SimpleNamespace(n=n, nz=nz, ntheta=nt, nscan=49, ndety=16)
    N, b = 3 * n // 2, lambda tag: bench.kernel_bytes(tag, slv)
    disc = lambda r: 8 * math.pi * r * r * nz
    obj, prj, smp = 8 * n * n * nz, 8 * nt * nz * n, 8 * nt * N * nz
    assert b("tomo_row_fwd") == obj + 8 * N * 2 * N * nz
    assert b("tomo_col_fwd") == pytest.approx(8 * N * 2 * N * nz + disc(N))
    assert b("tomo_gather") == pytest.approx(disc(N) + smp)
    assert b("tomo_line_idft") == smp + prj == b("tomo_adj_line")
    assert b("tomo_scatter") == pytest.approx(smp + disc(n))
    assert b("tomo_col_adj") == pytest.approx(disc(n) + 8 * n * 2 * n * nz)
    assert b("tomo_row_adj") == 8 * n * 2 * n * nz + obj
    assert b("tomo_scatter_fix") is None

"""bench.py on the CPU: its work models against the kernels they describe, and
its result line."""
import json
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


def test_result_line_is_short_strict_json():
    """A whole record of the default run (two traces of 100 iterations, seven
    seeds' comparisons, an unreached criterion) as one line under 8 KB that a
    strict parser reads, the measured values unrounded."""
    x = 0.12345678901234567
    crit = dict(criterion="c" * 140, plain_level=x, plain_s=x, plain_iters=91, warm_s=math.inf,
                warm_iters=None, speedup=x, plain_first_crossing_iters=91, network=x, after_short=x,
                warm_first_crossing_iters=8)
    run = dict(workload="w" * 50, iterations=100, lagrangian=dict(crit), object_error=dict(crit),
               fallback_to_plain=False)
    kern = {t: dict(avg_ms=x, algorithmic_bytes=x * 1e10, GB_s=x, frac_hbm=x) for t in bench.TAGS}
    out = dict(metric="m" * 70, value=x, unit="ADMM iters/s", n_gpus=1, steps=20, warmup=5,
               ms_per_step=1e3 * x, higher_is_better=True, scaling="weak", vs_baseline=None,
               dtype="c64", data="synthetic", config={f"key{i}": "v" * 10 for i in range(18)},
               roofline=dict(kern["ptycho_minf"], work={f"k{i}": x for i in range(10)}),
               kernels=kern, breakdown_ms_per_iter={t: x for t in bench.TAGS},
               operators={f"op{i}": {f"k{j}": x for j in range(6)} for i in range(4)},
               time_to_tol=dict(run, plain_trace={"e": [x] * 100, "l": [x] * 100},
                                warm_trace={"e": [x] * 100, "l": [x] * 100}),
               time_to_tol_warm128=dict(criterion="c" * 140, speedup_per_seed=[x] * 7,
                                        runs=[run] * 7),
               unet=dict(n=128, layers={f"l{i}": dict(cin=2, cout=16, ms=x, TFLOP_s=x,
                                                      frac_bf16_peak=x) for i in range(10)}),
               batch=dict(modes_s=dict(a=x, b=x, c=x)), cpu_baseline=dict(sample="s" * 330, value=x))
    line = bench.result_line(out)
    print(len(line))
    assert "\n" not in line and len(line) < 8000

    def no_constant(name):
        raise ValueError(name)
    res = json.loads(line, parse_constant=no_constant)
    assert res["value"] == x and res["ms_per_step"] == 1e3 * x
    assert set(res) == set(out)
    assert res["time_to_tol"]["lagrangian"]["warm_s"] is None
    assert res["unet"]["layers"]["l3"] == float(f"{x:.5g}")

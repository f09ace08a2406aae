"""The reverse sweep of the reflection rows' adjoint checked on the CPU against
forward-mode tangents of the same formulas, and the vertex adjoint's tangents
against 64 bits, on the device sources compiled as host C++ through a shim
(tests/cpu_geo/adjoint_check.cpp).

Both sides are float32 and round differently: each contraction multiplies a
few tens of rounded factors per bounce (1e-6 relative for five bounces), and
the slab's interior phase of a few tens of radians amplifies its rounding in
the material derivatives (1e-5). The bounds are five times that; the
degenerate rows put vectors of length near 1e-6 m through a normalization, at
coordinates rounded to 3e-5 m."""

from __future__ import annotations

import shutil
import subprocess
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent


@pytest.fixture(scope="module")
def report(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ is not available")
    exe = tmp_path_factory.mktemp("adjoint") / "adjoint_check"
    subprocess.run([gxx, "-O1", "-std=c++17", f"-I{HERE / 'cpu_geo'}", str(HERE / "cpu_geo" / "adjoint_check.cpp"),
                    "-o", str(exe)], check=True, capture_output=True, timeout=300)
    run = subprocess.run([str(exe)], check=True, capture_output=True, text=True, timeout=300)
    return [line.split() for line in run.stdout.splitlines()]


def test_no_row_is_nan(report):
    assert not [r for r in report if r[0] == "nan"]


@pytest.mark.parametrize("depth", [1, 2, 3, 4, 5])
def test_reflection_rows_adjoint_equals_tangents(report, depth):
    rows = [r for r in report if r[0] == str(depth)]
    assert len(rows) == 9
    for _, kind, ordinary, degenerate, masked in rows:
        assert float(ordinary) < (5.0e-5 if kind in ("eps", "sigma", "thickness") else 1.0e-5), kind
        assert float(degenerate) < 2.0e-4, kind
        assert int(masked) == 0, kind


@pytest.mark.parametrize("mode", ["coherent", "incoherent"])
@pytest.mark.parametrize("kind", ["planes", "wall_normals"])
def test_path_tangents_against_64_bits(report, mode, kind):
    """Against central differences in double. The interior phases of a path's
    float32 values move a derivative by 3e-5; an incoherent sum keeps only the
    amplitude's derivative, whose planes lose 1e-3 of it. The bounds are twice
    that."""
    error, = [float(r[2]) for r in report if r[:2] == [mode, kind]]
    assert error < (2.0e-3 if (mode, kind) == ("incoherent", "planes") else 6.0e-5)

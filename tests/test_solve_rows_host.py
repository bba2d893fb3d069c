"""The root finder's 8x8 solve (ipglasma_amd/csrc/solve_rows.hpp), built for the
host: against numpy.linalg.solve, with rows to exchange at every column, and what
the restart rule (a step above 1e5) sees of a singular system."""
import ctypes as C
import os
import shutil
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(HERE, "host", "solve_rows_host.cpp")
OUT = os.path.join(HERE, "_build", "libsolve_rows_host.so")
HIPCC = "/opt/rocm/bin/hipcc"
dp = np.ctypeslib.ndpointer(np.float64, flags="C")


@pytest.fixture(scope="module")
def solve():
    if not os.path.exists(HIPCC) and not shutil.which("hipcc"):
        pytest.skip("hipcc not available")
    os.makedirs(os.path.dirname(OUT), exist_ok=True)
    subprocess.run([HIPCC if os.path.exists(HIPCC) else "hipcc", "-x", "hip", "--offload-host-only", "-O2",
                    "-std=c++17", "-fPIC", "-shared", "-o", OUT, SRC], check=True, capture_output=True)
    f = C.CDLL(OUT).solve_rows_host
    f.argtypes = [dp] * 3

    def run(J, F):
        y = np.zeros(8)
        f(np.ascontiguousarray(J, dtype=float).reshape(-1), np.ascontiguousarray(F, dtype=float), y)
        return y
    return run


@pytest.mark.parametrize("kind", ["identity", "random", "reversed", "graded"])
def test_regular_systems(solve, kind):
    rng = np.random.default_rng(4)
    for _ in range(50):
        J = rng.normal(size=(8, 8))
        if kind == "identity":
            J = np.eye(8) + 0.1 * J
        elif kind == "reversed":  # the largest entry of every column in its last row
            J = np.eye(8)[::-1] + 0.1 * J
        elif kind == "graded":
            J = J * 10.0 ** -np.arange(8)[:, None]
        F = rng.normal(size=8)
        y = solve(J, F)
        # partial pivoting: backward error of ~8 eps times a growth of a few
        r = np.abs(J @ y - F)
        assert np.all(r <= 1e-13 * (np.abs(J) @ np.abs(y) + np.abs(F)))


def by_division(J, F):
    """the serial algorithm: Gaussian elimination, the first maximal pivot, rows
    divided by it unless it is zero"""
    J, F = J.copy(), F.copy()
    with np.errstate(all="ignore"):
        for j in range(7):
            p = j + int(np.argmax(np.abs(J[j:, j])))
            J[[j, p]], F[[j, p]] = J[[p, j]], F[[p, j]]
            if J[j, j] != 0:
                for r in range(j + 1, 8):
                    f = J[r, j] / J[j, j]
                    J[r] -= f * J[j]
                    F[r] -= f * F[j]
        y = np.zeros(8)
        for r in range(7, -1, -1):
            y[r] = (F[r] - sum(J[r, c] * y[c] for c in range(r + 1, 8))) / J[r, r]
    return y


@pytest.mark.parametrize("tiny", [0.0, 5e-324, 1e-310, 5e-309, 1e-306])
@pytest.mark.parametrize("col", range(8))
def test_singular_systems_restart_as_the_serial_algorithm(solve, tiny, col):
    """a column with nothing left but a pivot of zero or about the smallest normal
    number, and entries under it of half its size: its unknown's step is above
    1e5, which makes the link restart"""
    J = np.eye(8)
    J[col, col] = tiny
    J[col + 1:, col] = tiny / 2
    F = np.arange(1.0, 9.0)
    ref, y = by_division(J, F), solve(J, F)
    assert np.any(np.abs(ref) > 1e5)
    assert np.any(np.abs(y) > 1e5), y
    np.testing.assert_array_equal(np.isnan(y), np.isnan(ref))

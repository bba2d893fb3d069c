"""The reverse leapfrog step gathered per site (adjoint.hpp, what the kernels
run) against the same sums scattered with the per-site reverse functions that
test_adjoint_host.py checks by finite differences, on small clamped lattices:
every row and column is an edge or next to one.  The two add the same terms
(at most ~30 products of a few matrices of size ~3) in another order, so they
agree to 1e-13 of the largest cotangent."""
import ctypes as C
import os
import shutil
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(HERE, "host", "adjoint_gather_host.cpp")
OUT = os.path.join(HERE, "_build", "libadjoint_gather_host.so")
HIPCC = "/opt/rocm/bin/hipcc"
dp = np.ctypeslib.ndpointer(np.float64, flags="C")


@pytest.fixture(scope="module")
def lib():
    if not os.path.exists(HIPCC) and not shutil.which("hipcc"):
        pytest.skip("hipcc not available")
    os.makedirs(os.path.dirname(OUT), exist_ok=True)
    subprocess.run([HIPCC if os.path.exists(HIPCC) else "hipcc", "-x", "hip", "--offload-host-only", "-O2",
                    "-std=c++17", "-fPIC", "-shared", "-o", OUT, SRC], check=True, capture_output=True)
    L = C.CDLL(OUT)
    L.adj_gather_host.argtypes = [C.c_int, C.c_double, C.c_double, C.c_double] + [dp] * 8
    L.adj_link_update_host.argtypes = [dp, dp, C.c_double] + [dp] * 4
    return L


def store(a):
    return np.ascontiguousarray(np.stack([a.real, a.imag], -1).reshape(a.shape[0], 18))


def links(rng, n):
    return store(rng.normal(size=(n, 3, 3)) + 1j * rng.normal(size=(n, 3, 3)) + 2 * np.eye(3))


def hermitian(rng, n, traceless=False):
    a = rng.normal(size=(n, 3, 3)) + 1j * rng.normal(size=(n, 3, 3))
    a = (a + a.conj().transpose(0, 2, 1)) / 2
    if traceless:
        a = a - np.trace(a, axis1=1, axis2=2)[:, None, None] * np.eye(3) / 3
    return store(a)


@pytest.mark.parametrize("N", [2, 3, 4, 6])
def test_gathered_step_equals_scattered(lib, N):
    rng = np.random.default_rng(N)
    S = N * N
    ux, uy, phi = links(rng, S), links(rng, S), hermitian(rng, S)
    z1, z2, pib = hermitian(rng, S, True), hermitian(rng, S, True), hermitian(rng, S)
    out, ref = np.zeros((3, S, 18)), np.zeros((3, S, 18))
    lib.adj_gather_host(N, 0.7, 0.1, 2.0, ux, uy, phi, z1, z2, pib, out.reshape(-1), ref.reshape(-1))
    for k, name in enumerate(("Ux", "Uy", "phi")):
        err = np.abs(out[k] - ref[k]).max(axis=1).reshape(N, N)
        assert err.max() <= 1e-13 * np.abs(ref[k]).max(), (name, np.argwhere(err > 1e-12 * np.abs(ref[k]).max()))


def test_link_update(lib):
    rng = np.random.default_rng(5)
    for _ in range(20):
        u, e, yb, eb = links(rng, 1), hermitian(rng, 1, True), links(rng, 1), hermitian(rng, 1)
        out, ref = np.zeros((2, 18)), np.zeros((2, 18))
        lib.adj_link_update_host(u, e, 0.3, yb, eb, out.reshape(-1), ref.reshape(-1))
        np.testing.assert_allclose(out, ref, rtol=0, atol=1e-14 * np.abs(ref).max() * 20)

"""newton_polish: exact Newton steps after the root finder's stopping rule, in a
kernel of their own over the links that the plain root finder leaves."""
import time

import numpy as np
import pytest

import _cases as K
import _oracle as O
from test_gpu_parity import _GEN

pytestmark = pytest.mark.gpu


def _event(system, N, seed, **kw):
    import ipglasma_amd as I
    ev = I.Event(K.params(system, N=N, Ny=3, **kw), seed=seed)
    while not ev.init():
        pass
    return ev


@pytest.mark.parametrize("system,N", [("pPb", 16), ("AuAu", 48), ("pPb", 128)])
def test_polish_goes_on_from_the_plain_iterate(system, N):
    """a link that converged in the first pass (eight iterations at most) takes
    its plain iterations and n more, and moves by no more than the stopping
    level lets it; a straggling one (a Jacobian near singular) takes at least
    n more: a step that finds the residual above the stopping level again is
    not counted"""
    plain = _event(system, N, 5)
    it0, u0 = plain.newton_iterations(), [plain.field(k) for k in ("Ux", "Uy")]
    assert plain.observables()["newton_unconverged"] == 0
    plain.close()
    for n in (1, 4):
        ev = _event(system, N, 5, newton_polish=n)
        it = ev.newton_iterations()
        first = it0 <= 8
        assert first.mean() > 0.5  # the claim is about most links
        np.testing.assert_array_equal(it[first], it0[first] + n)
        assert np.all(it >= it0 + n)
        for k, u, f in zip(("Ux", "Uy"), u0, first.reshape(2, -1)):
            # Sum|F| <= 1e-6 and a Jacobian near the identity where links are near 1
            assert np.abs(ev.field(k) - u)[f].max() < 1e-5
        ev.close()


@pytest.mark.parametrize("system,N", [("pPb", 32), ("AuAu", 32), ("OO", 64)])
def test_polish_takes_links_to_round_off(system, N):
    """Sum|F_a| below 1e-13, the oracle's own bound: F is eight traces of products
    of matrices of norm 2 at most, ~5e-15 of round-off each way.  Four steps from
    1e-6 do it wherever the Jacobian's inverse is below ~100 (each step squares
    the distance, 1e-4 at most, up to a factor of that size)"""
    ev = _event(system, N, 5, newton_polish=4)
    S, idx = N * N, np.arange(N * N)
    V = [O.from_c(ev.field(k)) for k in ("VA", "VB")]
    nb = {"Ux": np.minimum(idx // N + 1, N - 1) * N + idx % N, "Uy": idx // N * N + np.minimum(idx % N + 1, N - 1)}
    for k, n in nb.items():
        U = O.from_c(ev.field(k))
        W = sum(v @ v[n].conj().transpose(0, 2, 1) for v in V)
        WU = W @ U.conj().transpose(0, 2, 1)
        M = W - W.conj().transpose(0, 2, 1) + WU - WU.conj().transpose(0, 2, 1)
        F = np.stack([-np.imag(np.trace(t @ M, axis1=1, axis2=2)) for t in _GEN], 1)
        J = np.stack([np.stack([-2 * np.real(np.trace(t @ WU @ u, axis1=1, axis2=2)) for u in _GEN], 1)
                      for t in _GEN], 1)
        fine = np.linalg.svd(J, compute_uv=False)[:, -1] > 0.01
        assert fine.mean() > 0.5
        assert np.abs(F).sum(1)[fine].max() < 1e-13, (k, np.sort(np.abs(F).sum(1)[fine])[-5:])
    ev.close()


def test_events_of_a_batch_polish_each_by_its_own_count():
    import ipglasma_amd as I
    pol = [0, 4, 0, 1]
    ps = [K.params("pPb", N=N, Ny=3, newton_polish=n) for N, n in zip((32, 48, 64, 32), pol)]
    plain = [K.params("pPb", N=N, Ny=3) for N in (32, 48, 64, 32)]
    it = []
    for q in (ps, plain):
        b = I.Batch(q, [3, 4, 5, 6])
        b.run()
        it.append([b.observables(e)["newton_iterations"] for e in range(4)])
        b.close()
    for a, c, N, n in zip(*it, (32, 48, 64, 32), pol):
        # exactly, but for a few stragglers' steps that are not counted
        assert 2 * N * N * n <= a - c <= 2 * N * N * n + (50 if n else 0)


def test_polish_costs_a_fraction_of_the_root_finder():
    """four steps without exponentials of the Jacobian's columns beside two to
    six with eight each; three times the plain call is far from both what they
    take (1.2 times) and what sending every link through the straggler kernel
    took (5 times)"""
    t = {}
    for n in (0, 4):
        ev = _event("PbPb", 256, 7, newton_polish=n)
        for _ in range(5):
            ev.init_fields()
        best = 1e9
        for _ in range(9):
            t0 = time.perf_counter()
            ev.init_fields()
            best = min(best, time.perf_counter() - t0)
        t[n] = best
        ev.close()
    assert t[4] < 3 * t[0], t

"""The long iterations make their x updates two at a time (gip_pcg.hip,
k_iter_dir): whatever iteration a solve stops at, x must hold every update.
One to six fixed iterations and a stop at each of a few tolerances, on both
long forms (more than 2^19 and more than 2^23 rows), with and without a
dictionary, against the oracle; the mixed solve with corrections after one,
two and three iterations; a breakdown in the second iteration.
"""
import time

import numpy as np
import pytest
import scipy.sparse as sp

from gip_amd import cavity, hip
from oracle import pyoracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    d = hip.Device(0)
    yield d
    d.close()


def _line(n, scale=None):
    """A shifted 1-D Laplacian (a few distinct rows: a dictionary), or one scaled row by row (none)."""
    T = sp.diags([-1.0, 2.05, -1.0], [-1, 0, 1], shape=(n, n)).tocsr()
    if scale is not None:
        S = sp.diags(scale)
        T = (S @ T @ S).tocsr()
    T.sort_indices()
    return T


@pytest.mark.parametrize("n,plain", [(2 ** 19 + 1, False), (2 ** 19 + 300, True), (2 ** 23 + 65, False)])
def test_x_holds_every_update(dev, n, plain):
    rng = np.random.default_rng(n)
    T = _line(n, 1.0 + 0.1 * rng.random(n) if plain else None)
    b, x0 = rng.standard_normal(n), 0.1 * rng.standard_normal(n)
    orc = pyoracle.Csr(T.indptr, T.indices, T.data, n)
    M = hip.Matrix(dev, T.indptr, T.indices, T.data, ncols=n, fp32=True)
    solver = hip.PCG(M, n)
    db, dx0, dx = dev.to_device(b), dev.to_device(x0), dev.array(n)
    for maxit in range(0, 7):
        r = solver.solve(db, dx, dx0, maxit=maxit)
        want, st, it, rel = pyoracle.pcg(orc, b, x0, n, maxit)
        assert r.iters == it == maxit and r.status == 0
        assert np.linalg.norm(dx.download() - want) <= 1e-12 * np.linalg.norm(want), maxit
    for tol in (0.5, 0.2, 0.1, 0.05, 0.02):
        r = solver.solve(db, dx, dx0, maxit=100, tol=tol, poll=3)
        want, st, it, rel = pyoracle.pcg(orc, b, x0, n, 100, tol=tol)
        assert r.iters == it and r.status == 0
        assert np.linalg.norm(dx.download() - want) <= 1e-12 * np.linalg.norm(want), tol
    for poll in (1, 2, 3):
        r = solver.solve(db, dx, dx0, maxit=200, tol=1e-10, precision=hip.PCG_MIXED, poll=poll)
        x = dx.download()
        print(f"[n={n} mixed poll {poll}] iters {r.iters} corrections {r.corrections}", flush=True)
        assert r.status == 0 and np.linalg.norm(b - T @ x) <= 1.01e-10 * np.linalg.norm(b)


@pytest.mark.parametrize("shape", [(96, 96, 64), (128, 256, 257)], ids=lambda s: "x".join(map(str, s)))
def test_cavity_iterates(dev, shape):
    c = cavity.generate(*shape, gamma=1e-3, ops=cavity.OP_BITS["L"])
    L, n, nall = c.op("L"), c.n_inner, c.n_all
    b = np.zeros(nall)
    b[:n] = cavity.rhs_normal(n, 4)
    x0 = np.zeros(nall)
    A = hip.Matrix.from_csr(dev, L)
    solver = hip.PCG(A, nall)
    dx, orc = dev.array(nall), pyoracle.Csr.of(L)
    for maxit in (1, 2, 3, 6):
        for precond in (True, False):
            r = solver.solve(dev.to_device(b), dx, dev.to_device(x0), maxit=maxit, precond=precond)
            assert r.iters == maxit
            if precond:
                want, st, it, rel = pyoracle.pcg(orc, b, x0, n, maxit)
                assert np.linalg.norm(dx.download() - want) <= 1e-12 * np.linalg.norm(want), maxit
    # a solver made before its operator's values changed keeps their diagonal
    A.set_values(2.0 * L.val)
    r = solver.solve(dev.to_device(b), dx, dev.to_device(x0), maxit=5)
    got = dx.download()
    F = hip.Matrix(dev, L.rowptr, L.col, 2.0 * L.val, nrows=n)
    fresh = hip.PCG(F, nall)
    fresh.solve(dev.to_device(b), dx, dev.to_device(x0), maxit=5)
    want = dx.download()
    assert np.linalg.norm(got - want) <= 1e-12 * np.linalg.norm(want)


def test_breakdown_keeps_the_updates_made(dev):
    """A solve that runs on after it has converged breaks down (p.Ap = 0) some
    iterations later: x is complete whatever parity it stops at."""
    n = 2 ** 19 + 64
    T = sp.identity(n, format="csr") * 2.0
    T = (T + sp.csr_matrix(([1.0, 1.0], ([0, 1], [1, 0])), shape=(n, n))).tocsr()
    T.sort_indices()
    M = hip.Matrix(dev, T.indptr, T.indices, T.data, ncols=n)
    solver = hip.PCG(M, n)
    b = np.ones(n)
    dx = dev.array(n)
    r = solver.solve(dev.to_device(b), dx, dev.to_device(np.zeros(n)), maxit=50, raise_on_breakdown=False)
    x = dx.download()
    print(f"[breakdown] iters {r.iters} status {r.status}", flush=True)
    assert np.all(np.isfinite(x))
    assert np.linalg.norm(b - T @ x) <= 1e-9 * np.linalg.norm(b)


# Mid-size operators: products in workgroups of 512 (up to 2^20 rows) or 1024
# rows, sweeps of four (up to 2^20) or eight rows per thread, and the forms on
# both sides of 2^21 rows; partial last workgroups.  A clustered mesh (no
# dictionary) in each layout, a uniform one with it; layouts agree bit for bit.
@pytest.mark.parametrize("beta", [0.0, 1.5])
@pytest.mark.parametrize("shape", [(128, 128, 64), (128, 128, 65), (128, 128, 128), (129, 128, 128)],
                         ids=lambda s: "x".join(map(str, s)))
def test_mid_size_forms(dev, shape, beta):
    c = cavity.generate(*shape, gamma=1e-3, ops=cavity.OP_BITS["L"], beta=beta)
    L, n, nall = c.op("L"), c.n_inner, c.n_all
    b = np.zeros(nall)
    b[:n] = cavity.rhs_normal(n, 4)
    x0 = np.zeros(nall)
    db, dx0, dx, orc = dev.to_device(b), dev.to_device(x0), dev.array(nall), pyoracle.Csr.of(L)
    want = {maxit: pyoracle.pcg(orc, b, x0, n, maxit)[0] for maxit in (1, 2, 5)}
    first = {}
    for fmt in (hip.FMT_AUTO, hip.FMT_ELL, hip.FMT_CSR):
        A = hip.Matrix(dev, L.rowptr, L.col, L.val, nrows=n, ncols=nall, fmt=fmt, fp32=True)
        solver = hip.PCG(A, nall)
        for maxit in (1, 2, 5):
            for precision in (hip.PCG_FP64, hip.PCG_MIXED):
                r = solver.solve(db, dx, dx0, maxit=maxit, precision=precision)
                x = dx.download()
                assert r.iters == maxit
                if precision == hip.PCG_FP64:
                    assert np.linalg.norm(x - want[maxit]) <= 1e-12 * np.linalg.norm(want[maxit]), (fmt, maxit)
                assert np.array_equal(first.setdefault((maxit, precision), x), x), (fmt, maxit, precision)
        del solver, A


def _band(n, kinds):
    """A shifted 7-diagonal Laplacian, scaled symmetrically by `kinds` factors in turn: as many tuples and the few
    of its ends; more than two tuples in a slice from three factors on."""
    s = 1.0 + 0.05 * (np.arange(n) % kinds)
    diags = [-(s[k:] * s[:n - k]) for k in (9, 3, 1)]
    T = sp.diags(diags + [6.15 * s * s] + diags[::-1], [-9, -3, -1, 0, 1, 3, 9], shape=(n, n)).tocsr()
    T.sort_indices()
    return T


# The long iterations with the dictionary and without: s formed again from r
# (FP64, and FP32 where no slice needs ids) or stored, ids or scalar tuples.
@pytest.mark.parametrize("dictionary,kinds", [(True, 1), (True, 5), (False, 5)])
@pytest.mark.parametrize("n", [2 ** 19 + 300, 2 ** 21 + 1, 2 ** 23 + 65])
def test_x_holds_every_update_with_the_dictionary(dev, n, dictionary, kinds):
    rng = np.random.default_rng(n)
    T = _band(n, kinds)
    b, x0 = rng.standard_normal(n), 0.1 * rng.standard_normal(n)
    orc = pyoracle.Csr(T.indptr, T.indices, T.data, n)
    M = hip.Matrix(dev, T.indptr, T.indices, T.data, ncols=n, fp32=True, dictionary=dictionary)
    # the two end slices hold more tuples than two whatever the factors
    assert M.info()["format"] == hip.FMT_STENCIL and (M.dict_state()[0] != 0) == dictionary
    assert not dictionary or M.dict_state()[1] <= 40
    solver = hip.PCG(M, n)
    db, dx0, dx = dev.to_device(b), dev.to_device(x0), dev.array(n)
    for maxit in (1, 2, 3, 4):
        for precond in (True, False):
            r = solver.solve(db, dx, dx0, maxit=maxit, precond=precond)
            assert r.iters == maxit and r.status == 0
            if precond:
                want, st, it, rel = pyoracle.pcg(orc, b, x0, n, maxit)
                assert np.linalg.norm(dx.download() - want) <= 1e-12 * np.linalg.norm(want), maxit
    for tol in (0.2, 0.1, 0.05):
        r = solver.solve(db, dx, dx0, maxit=100, tol=tol, poll=3)
        want, st, it, rel = pyoracle.pcg(orc, b, x0, n, 100, tol=tol)
        assert r.iters == it and r.status == 0
        assert np.linalg.norm(dx.download() - want) <= 1e-12 * np.linalg.norm(want), tol
    for poll in (1, 2, 3):
        r = solver.solve(db, dx, dx0, maxit=200, tol=1e-10, precision=hip.PCG_MIXED, poll=poll)
        x = dx.download()
        assert r.status == 0 and np.linalg.norm(b - T @ x) <= 1.01e-10 * np.linalg.norm(b)


# Exact breakdowns: with the eigenvalue 2 (Jacobi: 1) the first iteration, with
# 1 and 3 in equal numbers the second leaves r = 0 to the last bit, so the one
# after stops at p.Ap = 0, an odd and an even number of iterations done (every
# sum is one of multiples of 1/16 below 2^24: exact in any order).
@pytest.mark.parametrize("form", ["dictionary", "stencil", "ell", "csr"])
@pytest.mark.parametrize("n", [2 ** 19 + 64, 2 ** 21 + 64, 2 ** 23 + 64])
@pytest.mark.parametrize("iters", [1, 2])
def test_breakdown_after_an_odd_and_an_even_iteration(dev, n, form, iters):
    diag = np.full(n, 2.0) if iters == 1 else np.where(np.arange(n) % 2, 3.0, 1.0)
    col = np.arange(n)[:, None] + np.array([-9, -3, -1, 0, 1, 3, 9])[None, :]
    inside = (col >= 0) & (col < n)
    val = np.zeros((n, 7))
    val[:, 3] = diag
    rowptr = np.concatenate([[0], np.cumsum(inside.sum(1))])
    M = hip.Matrix(dev, rowptr, col[inside], val[inside], ncols=n, dictionary=form == "dictionary",
                   fmt={"ell": hip.FMT_ELL, "csr": hip.FMT_CSR}.get(form, hip.FMT_STENCIL))
    assert (M.dict_state()[0] != 0) == (form == "dictionary")
    solver = hip.PCG(M, n)
    dx = dev.array(n)
    for tol, poll in ((0.0, 16), (1e-300, 1), (1e-300, 16)):
        r = solver.solve(dev.to_device(np.ones(n)), dx, dev.to_device(np.zeros(n)), maxit=50, tol=tol, poll=poll,
                         precond=iters == 1, raise_on_breakdown=False)
        if tol:  # r.r = 0 meets any tolerance: no breakdown, the same x
            assert r.status == hip.OK and r.iters == iters
        else:
            assert r.status == hip.EBREAKDOWN and r.iters == iters
        assert np.abs(dx.download() * diag - 1.0).max() <= 2e-16 * (iters - 1)


@pytest.mark.parametrize("n", [4096, 2 ** 19 + 64])
def test_a_long_fixed_run_ends_soon_after_a_breakdown(dev, n):
    """200,000 iterations, of which the first breaks down: the host reads the state every 4096."""
    rowptr = np.arange(n + 1)
    M = hip.Matrix(dev, rowptr, np.arange(n), np.full(n, 2.0), ncols=n, fmt=hip.FMT_CSR)
    solver, dx = hip.PCG(M, n), dev.array(n)
    b, z = dev.to_device(np.ones(n)), dev.to_device(np.zeros(n))
    solver.solve(b, dx, z, maxit=2, raise_on_breakdown=False)
    t0 = time.perf_counter()
    r = solver.solve(b, dx, z, maxit=200000, raise_on_breakdown=False)
    took = time.perf_counter() - t0
    print(f"[long fixed run {n}] {1e3 * took:.1f} ms", flush=True)
    assert r.status == hip.EBREAKDOWN and r.iters == 1
    assert np.array_equal(dx.download(), np.full(n, 0.5))
    assert took < 0.3
    # and one without a breakdown runs through its reads of the state
    L = _line(n)
    M = hip.Matrix(dev, L.indptr, L.indices, L.data, ncols=n)
    solver = hip.PCG(M, n)
    c = np.random.default_rng(3).standard_normal(n)
    r = solver.solve(dev.to_device(c), dx, z, maxit=4100, raise_on_breakdown=False)
    if r.status == 0:
        assert r.iters == 4100
    assert np.linalg.norm(c - L @ dx.download()) <= 1e-12 * np.linalg.norm(c)

"""The symmetric form of a stencil operator's slot values in the FP64 PCG's
product (include/gip_hip.h, GIP_MAT_NO_SYM; gip_layout.h, plan_symmetric):
a slot of offset -d reads row r - d's slot of offset +d, so the product
must give the full layout's bits.  Checked against the same operator built
without it (GIP_MAT_NO_SYM): FP64 iterates bitwise on both long iteration
forms (more and fewer than 2^23 rows) and for 7- and 8-slot layouts (128^3
and 96^3, whose boundary slices pick an eighth offset), a tolerance stop,
the clustered mesh, the mixed solve untouched (its FP32 product keeps all
slots); after a change of
values the form is made again (scaled values) or refused (one value off
by one unit in the last place), and the solve still equals the full one.
"""
import time

import numpy as np
import pytest

from gip_amd import cavity, hip

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    d = hip.Device(0)
    yield d
    d.close()


def _case(nx, ny=None, nz=None, beta=0.0):
    c = cavity.generate(nx, ny, nz, beta=beta, gamma=1e-3, ops=cavity.OP_BITS["L"])
    b = np.zeros(c.n_all)
    b[:c.n_inner] = cavity.rhs_normal(c.n_inner, 11)
    return c, c.op("L"), b


def _solve(dev, A, c, b, **kw):
    solver = hip.PCG(A, c.n_all)
    dx = dev.array(c.n_all)
    r = solver.solve(dev.to_device(b), dx, dev.to_device(np.zeros(c.n_all)), **kw)
    x = dx.download()
    solver.destroy()
    return r, x


def _pair(dev, L, **kw):
    A = hip.Matrix.from_csr(dev, L, **kw)
    F = hip.Matrix.from_csr(dev, L, sym=False, **kw)
    assert A.info()["format"] == hip.FMT_STENCIL and F.info()["format"] == hip.FMT_STENCIL
    return A, F


@pytest.mark.parametrize("shape", [(96, 96, 96), (128, 128, 128), (256, 256, 129)],
                         ids=["96^3", "128^3", "256x256x129"])
def test_fp64_fixed_iterations_bitwise(dev, shape):
    c, L, b = _case(*shape)
    print(f"[sym fp64 {shape}] rows {c.n_inner}", flush=True)
    A, F = _pair(dev, L)
    assert A.sym_state()[0] == 2 and F.sym_state()[0] == 0
    ra, xa = _solve(dev, A, c, b, maxit=40)
    rf, xf = _solve(dev, F, c, b, maxit=40)
    st, b64 = A.sym_state()
    print(f"[sym fp64 {shape}] state {st} bytes {b64} (full layout {F.product_bytes()}) relres {ra.relres:.6e}",
          flush=True)
    assert st == 1 and F.sym_state()[0] == 0
    assert 0 < b64 < 0.8 * F.product_bytes()
    assert ra.iters == rf.iters == 40 and ra.relres == rf.relres
    assert np.array_equal(xa, xf)
    A.destroy()
    F.destroy()


def test_fp64_tolerance_stop_bitwise_and_mixed_untouched(dev):
    """A tolerance-stopped FP64 solve equals the full one bitwise; the mixed
    solve (whose FP32 product keeps all slots) neither makes nor needs the
    form and equals the full operator's mixed solve bitwise."""
    c, L, b = _case(128)
    A, F = _pair(dev, L, fp32=True)
    kw = dict(maxit=20000, tol=1e-10, precision=hip.PCG_MIXED, poll=32)
    ra, xa = _solve(dev, A, c, b, **kw)
    rf, xf = _solve(dev, F, c, b, **kw)
    print(f"[sym mixed 128^3] iters {ra.iters}/{rf.iters} corrections {ra.corrections}/{rf.corrections}", flush=True)
    assert A.sym_state()[0] == 2
    assert ra.status == rf.status == 0
    assert (ra.iters, ra.corrections) == (rf.iters, rf.corrections)
    assert np.array_equal(xa, xf)
    kw = dict(maxit=5000, tol=1e-6)
    ra, xa = _solve(dev, A, c, b, **kw)
    rf, xf = _solve(dev, F, c, b, **kw)
    print(f"[sym fp64 128^3 tol 1e-6] iters {ra.iters}/{rf.iters}", flush=True)
    assert A.sym_state()[0] == 1
    assert ra.status == rf.status == 0 and ra.iters == rf.iters
    assert np.array_equal(xa, xf)
    A.destroy()
    F.destroy()


def test_clustered_mesh_bitwise(dev):
    c, L, b = _case(128, beta=1.5)
    A, F = _pair(dev, L)
    ra, xa = _solve(dev, A, c, b, maxit=30)
    rf, xf = _solve(dev, F, c, b, maxit=30)
    assert A.sym_state()[0] == 1
    assert np.array_equal(xa, xf)
    A.destroy()
    F.destroy()


def test_changed_values_remake_or_refuse_the_form(dev):
    c, L, b = _case(96, 96, 80)
    A = hip.Matrix.from_csr(dev, L)
    _solve(dev, A, c, b, maxit=5)
    assert A.sym_state()[0] == 1
    # scaled values stay symmetric: the form is made again at the next solve
    v2 = L.val * 2.0
    A.set_values(v2)
    assert A.sym_state()[0] == 2
    F = hip.Matrix(dev, L.rowptr, L.col, v2, nrows=L.nrows, sym=False)
    ra, xa = _solve(dev, A, c, b, maxit=25)
    rf, xf = _solve(dev, F, c, b, maxit=25)
    assert A.sym_state()[0] == 1
    assert np.array_equal(xa, xf)
    F.destroy()
    # one off-diagonal value of an interior row one unit in the last place
    # lower: no longer symmetric, the solve falls back to the full values
    v3 = v2.copy()
    r0 = 96 * 96 * 40 + 96 * 48 + 48
    j = [j for j in range(L.rowptr[r0], L.rowptr[r0 + 1]) if L.col[j] == r0 + 96][0]
    v3[j] = np.nextafter(v3[j], 0.0)
    A.set_values(v3)
    F = hip.Matrix(dev, L.rowptr, L.col, v3, nrows=L.nrows, sym=False)
    ra, xa = _solve(dev, A, c, b, maxit=25)
    rf, xf = _solve(dev, F, c, b, maxit=25)
    print(f"[sym values changed] state {A.sym_state()[0]}", flush=True)
    assert A.sym_state()[0] == -1
    assert np.array_equal(xa, xf)
    A.destroy()
    F.destroy()


def test_no_arrays_beside_a_dictionary(dev):
    """A solve that multiplies from the dictionary neither makes nor keeps the symmetric arrays (100 MB here)."""
    torch = pytest.importorskip("torch")
    c, L, b = _case(128)
    A = hip.Matrix.from_csr(dev, L)
    assert A.dict_state()[0] != 0
    solver = hip.PCG(A, c.n_all)
    db, dx, dz = dev.to_device(b), dev.array(c.n_all), dev.to_device(np.zeros(c.n_all))

    def grown(call, want):
        """Whether `call` changed the memory in use by want(bytes); the driver may count freed memory a little later."""
        dev.sync()
        free = torch.cuda.mem_get_info()[0]
        call()
        for _ in range(40):
            if want(free - torch.cuda.mem_get_info()[0]):
                return True
            time.sleep(0.05)
        return False

    def solve():
        solver.solve(db, dx, dz, maxit=3)

    def symmetric():
        assert A.sym_state()[0] == 1

    def little(bytes_):
        return abs(bytes_) < 16 << 20

    assert grown(solve, little)
    A.set_values(2.0 * L.val)
    assert grown(solve, little)
    # asked for, the symmetry is checked, and the arrays go again
    assert grown(symmetric, little)
    # without the dictionary (no two rows alike, still symmetric) the solve makes them; with it back they go
    row = np.repeat(np.arange(L.nrows), np.diff(L.rowptr))
    s = 1.0 + 0.1 * np.random.default_rng(5).random(c.n_all)
    v = (s[row] * s[L.col]) * L.val
    A.set_values(v)
    assert A.dict_state()[0] == 0
    assert grown(solve, lambda m: m > 64 << 20)
    symmetric()
    assert grown(lambda: A.set_values(L.val), lambda m: m < -(32 << 20))
    assert A.sym_state()[0] == 2
    assert grown(solve, little)
    symmetric()


@pytest.mark.parametrize("beta", [0.0, 1.5])
@pytest.mark.parametrize("shape", [(96, 96, 96), (128, 128, 64), (128, 128, 128), (113, 128, 150), (144, 128, 128),
                                   (256, 256, 129), (208, 200, 208)], ids=lambda s: "x".join(map(str, s)))
def test_the_form_itself_bitwise(dev, shape, beta):
    """Operators without a dictionary, whose FP64 products do read the form: 7 and 8 slots, workgroups of 512, 1024
    and 256 rows, and the row-per-thread iteration past 2^23 rows."""
    c, L, b = _case(*shape, beta=beta)
    A, F = _pair(dev, L, dictionary=False)
    for kw in (dict(maxit=15), dict(maxit=400, tol=1e-2)):
        ra, xa = _solve(dev, A, c, b, **kw)
        rf, xf = _solve(dev, F, c, b, **kw)
        assert A.dict_state()[0] == 0 and A.sym_state()[0] == 1 and F.sym_state()[0] == 0
        print(f"[sym form {shape} beta {beta}] iters {ra.iters}", flush=True)
        assert ra.iters == rf.iters and ra.relres == rf.relres
        assert np.array_equal(xa, xf)
    # one value off by one unit in the last place: the full product, not the form
    v = L.val.copy()
    r0 = L.nrows // 2 + 3
    j = [j for j in range(L.rowptr[r0], L.rowptr[r0 + 1]) if r0 < L.col[j] < L.nrows][0]
    v[j] = np.nextafter(v[j], 0.0)
    A.set_values(v)
    F.set_values(v)
    ra, xa = _solve(dev, A, c, b, maxit=15)
    rf, xf = _solve(dev, F, c, b, maxit=15)
    assert A.sym_state()[0] == -1
    assert np.array_equal(xa, xf)

"""The dictionary of a stencil operator's slot values (gip_dict.hip): from
2^18 rows on, an operator whose rows repeat a few value tuples is multiplied
from the distinct tuples.  The values are the stored ones bit for bit, so
every product must equal the CSR layout's bitwise: at the smallest size, on
meshes whose lines fill slices (scalar tuples), straddle them (per-row ids)
and end in a partial slice, for the operators of every shape, after changes
of the values (made again, one value off, no repetition left, rebuilt on the
device), and in FP32.
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


def _products(dev, A, C, seed, fp32=False):
    """y = A x and y = a A x + b y over random x, both layouts, bitwise."""
    rng = np.random.default_rng(seed)
    m, n = A.cols_needed, A.nrows
    dx = dev.to_device(rng.standard_normal(m))
    y0 = rng.standard_normal(n)
    for op in (lambda M, y: M.spmv(dx, y), lambda M, y: M.spmv_ab(dx, y, -1.25, 0.5)):
        got, want = dev.to_device(y0), dev.to_device(y0)
        op(A, got)
        op(C, want)
        assert np.array_equal(got.download(), want.download())
    if fp32:
        sx = dev.to_device(rng.standard_normal(m).astype(np.float32))
        got, want = dev.array(n, np.float32), dev.array(n, np.float32)
        A.spmv32(sx, got)
        C.spmv32(sx, want)
        assert np.array_equal(got.download(), want.download())


@pytest.mark.parametrize("shape", [(64, 64, 64), (64, 64, 63), (128, 64, 33), (63, 65, 67), (97, 97, 97),
                                   (256, 32, 40), (129, 130, 16), (192, 48, 48)],
                         ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("beta", [0.0, 1.5])
def test_laplacian_products_bitwise(dev, shape, beta):
    c = cavity.generate(*shape, beta=beta, gamma=1e-3, ops=cavity.OP_BITS["L"])
    L = c.op("L")
    print(f"[dictionary {shape} beta {beta}] rows {L.nrows}", flush=True)
    A = hip.Matrix.from_csr(dev, L, fp32=True)
    C = hip.Matrix.from_csr(dev, L, fmt=hip.FMT_CSR, fp32=True)
    assert A.info()["format"] == hip.FMT_STENCIL
    assert np.array_equal(A.values(), L.val)
    _products(dev, A, C, 1, fp32=True)


@pytest.mark.parametrize("n", [64, 72])
def test_every_operator_bitwise(dev, n):
    c = cavity.generate(n, gamma=1e-3)
    for name in cavity.OPS:
        op = c.op(name)
        print(f"[dictionary {name} {n}^3] rows {op.nrows}", flush=True)
        A, C = hip.Matrix.from_csr(dev, op), hip.Matrix.from_csr(dev, op, fmt=hip.FMT_CSR)
        _products(dev, A, C, 2)
        # the transposed product refreshes its operator's values on each call
        if name in ("D", "Gx", "SO"):
            x = dev.to_device(np.random.default_rng(3).standard_normal(A.nrows))
            cols = max(A.cols_needed, C.cols_needed)
            got, want = dev.array(cols), dev.array(cols)
            for M, y in ((A, got), (C, want)):
                M.spmv_t(x, y, cols)
            assert np.array_equal(got.download(), want.download())
            v = op.val * 1.5
            A.set_values(v)
            C.set_values(v)
            for M, y in ((A, got), (C, want)):
                M.spmv_t(x, y, cols)
            assert np.array_equal(got.download(), want.download())
        A.destroy()
        C.destroy()


@pytest.mark.parametrize("n", [64, 66])
def test_changed_values(dev, n):
    c = cavity.generate(n, gamma=1e-3)
    L = c.op("L")
    A = hip.Matrix.from_csr(dev, L, fp32=True)
    C = hip.Matrix.from_csr(dev, L, fmt=hip.FMT_CSR, fp32=True)
    rng = np.random.default_rng(4)
    one = L.val.copy()
    one[L.nnz // 2] = np.nextafter(one[L.nnz // 2], 0.0)
    signs = np.where(rng.random(L.nnz) < 0.5, -0.0, L.val)  # zeros of both signs, many tuples
    for v in (2.0 * L.val, one, rng.standard_normal(L.nnz), signs, L.val):
        A.set_values(v)
        C.set_values(v)
        assert np.array_equal(A.values(), v)
        _products(dev, A, C, 5, fp32=True)
    # values rebuilt on the device by a product: the dictionary made before is stale
    D = c.op("D")
    A, C = hip.Matrix.from_csr(dev, D), hip.Matrix.from_csr(dev, D, fmt=hip.FMT_CSR)
    E = hip.Matrix.from_csr(dev, c.op("Ec"))
    mf = dev.to_device(rng.standard_normal(c.n_faces))
    for M in (A, C):
        E.spmv_vals(mf, M)
    _products(dev, A, C, 6)
    assert np.array_equal(A.values(), C.values())


def test_captured_products_follow_the_values(dev):
    """A graph that holds a product or a change of values, replayed after the values changed otherwise."""
    import torch

    c = cavity.generate(64, gamma=1e-3, ops=cavity.OP_BITS["L"])  # 2^18 rows: a dictionary
    L, n, nall = c.op("L"), c.n_inner, c.n_all
    A = hip.Matrix.from_csr(dev, L, fp32=True)
    C = hip.Matrix.from_csr(dev, L, fmt=hip.FMT_CSR)
    nnz = L.val.size
    ident = hip.Matrix(dev, np.arange(nnz + 1), np.arange(nnz), np.ones(nnz), ncols=nnz, fmt=hip.FMT_CSR)
    rng = np.random.default_rng(0)
    dx, sx = dev.to_device(rng.standard_normal(nall)), dev.to_device(rng.standard_normal(nall).astype(np.float32))
    dv = dev.to_device(5.0 * L.val)
    y, s, want, swant = dev.array(n), dev.array(n, np.float32), dev.array(n), dev.array(n, np.float32)
    stream = torch.cuda.ExternalStream(hip.lib().gip_stream(dev.ctx))
    product, change = torch.cuda.CUDAGraph(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(product, stream=stream, capture_error_mode="thread_local"):
        A.spmv(dx, y)
        A.spmv32(sx, s)

    def replayed():
        with torch.cuda.stream(stream):
            product.replay()
        return y.download(), s.download()

    def eager(M):
        M.spmv(dx, want)
        return want.download()

    A.spmv32(sx, swant)
    base, base32 = eager(C), swant.download()
    for factor in (1.0, 2.0, 0.5, 4.0):
        A.set_values(factor * L.val)
        assert np.array_equal(eager(A), factor * base)
        for _ in range(2):
            got, got32 = replayed()
            assert np.array_equal(got, factor * base) and np.array_equal(got32, np.float32(factor) * base32)
    with torch.cuda.graph(change, stream=stream, capture_error_mode="thread_local"):
        ident.spmv_vals(dv, A)
    C.set_values(5.0 * L.val)
    five = eager(C)
    for _ in range(2):
        A.set_values(L.val)
        assert np.array_equal(eager(A), base)
        with torch.cuda.stream(stream):
            change.replay()
        assert np.array_equal(eager(A), five) and np.array_equal(replayed()[0], five)


# ---- which operators have one -------------------------------------------------

OFFSETS7 = (-9, -3, -1, 0, 1, 3, 9)
OFFSETS8 = (-9, -3, -1, 0, 1, 3, 9, 27)


def band(n, rows, offsets=OFFSETS7):
    """CSR arrays of a band operator whose row r holds the values rows[r] at columns r + offsets (inside the
    operator), the number of distinct rows with zeros for the missing entries (the dictionary's tuples, since
    every slice of 64 rows has the same slots) and whether a slice holds more than two of them."""
    col = np.arange(n)[:, None] + np.asarray(offsets)[None, :]
    inside = (col >= 0) & (col < n)
    kinds, kind = np.unique(np.where(inside, rows, 0.0), axis=0, return_inverse=True)
    k = np.sort(np.concatenate([kind.ravel(), np.full(-n % 64, kind.ravel()[-1])]).reshape(-1, 64), axis=1)
    many = bool((np.diff(k, axis=1) != 0).sum(1).max() > 1)
    rowptr = np.concatenate([[0], np.cumsum(inside.sum(1))]).astype(np.int32)
    return rowptr, col[inside].astype(np.int32), np.ascontiguousarray(rows[inside]), kinds.shape[0], many


def pick(n, k, seed, by=1):
    """Row indices into k kinds, drawn anew every `by` rows, the first row of every kind somewhere."""
    return np.repeat(np.random.default_rng(seed).integers(0, k, -(-n // by)), by)[:n]


@pytest.mark.parametrize("n", [2 ** 18 + 1, 2 ** 20 - 37])
@pytest.mark.parametrize("offsets", [(-1, 0, 1), OFFSETS7, OFFSETS8], ids=lambda o: f"{len(o)} slots")
@pytest.mark.parametrize("kinds,by", [(1, 1), (2, 1), (3, 64), (40, 1), (3000, 64)])
def test_tuples_of_a_band(dev, n, offsets, kinds, by):
    """The number of tuples, whether slices need their rows' numbers, and the products."""
    rng = np.random.default_rng(7)
    which = pick(n, kinds, 8, by)
    rowptr, col, val, tuples, many = band(n, rng.standard_normal((kinds, len(offsets)))[which], offsets)
    print(f"[tuples n {n} slots {len(offsets)} kinds {kinds} by {by}] {tuples}", flush=True)
    A = hip.Matrix(dev, rowptr, col, val, nrows=n, ncols=n, fp32=True)
    C = hip.Matrix(dev, rowptr, col, val, nrows=n, ncols=n, fmt=hip.FMT_CSR, fp32=True)
    state, got, nbytes = A.dict_state()
    assert got == tuples and state == (2 if many else 1)
    assert 16 * n < nbytes < A.product_bytes()
    assert C.dict_state() == (0, 0, 0)
    _products(dev, A, C, 9, fp32=True)


def test_states(dev):
    """64-row slices of one tuple need no numbers; values changed on the device, or without repetition, have no
    dictionary until values are set that do."""
    n = 2 ** 18 + 640
    rng = np.random.default_rng(1)
    rowptr, col, val, tuples, _ = band(n, np.tile(rng.standard_normal(3), (n, 1)), (-64, 0, 64))
    A = hip.Matrix(dev, rowptr, col, val, nrows=n, ncols=n)
    assert A.dict_state()[:2] == (1, tuples) and tuples == 3
    A.set_values(rng.standard_normal(val.size))
    assert A.dict_state() == (0, 0, 0)
    A.set_values(val)
    assert A.dict_state()[:2] == (1, 3)
    nnz = val.size
    ident = hip.Matrix(dev, np.arange(nnz + 1), np.arange(nnz), np.ones(nnz), ncols=nnz, fmt=hip.FMT_CSR)
    ident.spmv_vals(dev.to_device(2.0 * val), A)
    assert A.dict_state() == (0, 0, 0)
    A.set_values(val)
    assert A.dict_state()[:2] == (1, 3)


@pytest.mark.parametrize("shape,state", [((128, 64, 33), 1), ((65, 64, 64), 2), ((97, 97, 97), 2)],
                         ids=lambda s: "x".join(map(str, s)) if isinstance(s, tuple) else str(s))
def test_uniform_meshes_have_one(dev, shape, state):
    c = cavity.generate(*shape, gamma=1e-3, ops=cavity.OP_BITS["L"])
    A = hip.Matrix.from_csr(dev, c.op("L"), fp32=True)
    got, tuples, nbytes = A.dict_state()
    print(f"[dictionary {shape}] state {got} tuples {tuples} bytes {nbytes} of {A.product_bytes()}", flush=True)
    assert got == state and 0 < tuples <= c.n_inner // 8
    assert nbytes < 0.5 * A.product_bytes() and A.dict_state(fp32=True)[2] < nbytes
    # clustered: no two lines alike
    c = cavity.generate(*shape, beta=1.5, gamma=1e-3, ops=cavity.OP_BITS["L"])
    assert hip.Matrix.from_csr(dev, c.op("L")).dict_state() == (0, 0, 0)


@pytest.mark.parametrize("shape", [(72, 64, 64), (128, 128, 128)], ids=lambda s: "x".join(map(str, s)))
def test_setting_values_costs_little_more_with_a_dictionary(dev, shape):
    """Making the dictionary anew adds 0.1 to 0.2 ms to gip_mat_set_values here (with every row at the table for
    itself, and memory allocated for it, 1.1 and 2.8), beside the same values in a layout without one."""
    c = cavity.generate(*shape, gamma=1e-3, ops=cavity.OP_BITS["L"])
    L = c.op("L")
    A, E = hip.Matrix.from_csr(dev, L), hip.Matrix.from_csr(dev, L, fmt=hip.FMT_ELL)
    assert A.dict_state()[0] != 0 and E.dict_state()[0] == 0
    best = []
    for M in (A, E):
        times = []
        for _ in range(15):
            dev.sync()
            t0 = time.perf_counter()
            M.set_values(L.val)
            dev.sync()
            times.append(time.perf_counter() - t0)
        best.append(min(times))
    print(f"[set_values {shape}] {1e3 * best[0]:.2f} ms, ELL {1e3 * best[1]:.2f}", flush=True)
    assert best[0] - best[1] < 0.7e-3


def lines_per_slice(which):
    """Mean over the 64-row slices of the cache lines of 16 tuples that a slice of more than two tuples gathers
    from, the tuples numbered by the first row that holds them (rows without all their entries left out)."""
    _, first, kind = np.unique(which, return_index=True, return_inverse=True)
    number = np.argsort(np.argsort(first))[kind]
    slices = [np.unique(number[s:s + 64]) for s in range(0, which.size, 64)]
    return sum(np.unique(own // 16).size for own in slices if own.size > 2) / len(slices)


@pytest.mark.parametrize("kinds,by,fp64,fp32", [(100, 1, True, True), (300, 1, True, False), (5000, 1, False, False),
                                                (20000, 1, False, False), (20000, 64, True, True),
                                                (20000, 8, True, True)])
def test_scattered_tuples_are_multiplied_as_stored(dev, kinds, by, fp64, fp32):
    """Gathers from more than 32 cache lines per slice and slot (FP32: 12) would take longer than the stored values."""
    n = 5 * 2 ** 18  # FP32 products read ids from here on
    which = pick(n, kinds, 11, by)
    col = np.arange(n)[:, None] + np.asarray(OFFSETS7)[None, :]
    inside = (col >= 0) & (col < n)
    rowptr = np.concatenate([[0], np.cumsum(inside.sum(1))])
    col, val = col[inside], np.random.default_rng(12).standard_normal((kinds, 7))[which][inside]
    A = hip.Matrix(dev, rowptr, col, val, nrows=n, ncols=n, fp32=True)
    C = hip.Matrix(dev, rowptr, col, val, nrows=n, ncols=n, fmt=hip.FMT_CSR, fp32=True)
    lines = lines_per_slice(which)
    print(f"[scattered kinds {kinds} by {by}] {lines:.1f} lines per slice, state {A.dict_state()[0]}", flush=True)
    assert fp64 == (lines <= 32) and fp32 == (lines <= 12)
    assert (A.dict_state()[0] != 0) == fp64
    assert (A.dict_state(fp32=True)[0] != 0) == fp32
    _products(dev, A, C, 13, fp32=True)


@pytest.mark.parametrize("shape,fp32", [((64, 64, 65), False), ((128, 64, 64), False), ((97, 97, 97), False),
                                        ((104, 104, 104), False), ((128, 128, 64), True), ((112, 112, 112), True)],
                         ids=lambda s: "x".join(map(str, s)) if isinstance(s, tuple) else str(s))
def test_fp32_products_that_fit_the_caches_read_the_stored_values(dev, shape, fp32):
    c = cavity.generate(*shape, gamma=1e-3, ops=cavity.OP_BITS["L"])
    A = hip.Matrix.from_csr(dev, c.op("L"), fp32=True)
    assert A.dict_state()[0] != 0 and (A.dict_state(fp32=True)[0] != 0) == fp32
    _products(dev, A, hip.Matrix.from_csr(dev, c.op("L"), fmt=hip.FMT_CSR, fp32=True), 14, fp32=True)


def test_no_dictionary_where_nothing_reads_one(dev):
    """Turned off; five slots, which have no kernel for it; values that a captured graph may change, set again."""
    c = cavity.generate(72, gamma=1e-3, ops=cavity.OP_BITS["L"])
    L = c.op("L")
    A, D = hip.Matrix.from_csr(dev, L, dictionary=False), hip.Matrix.from_csr(dev, L)
    assert A.dict_state() == (0, 0, 0) and D.dict_state()[0] != 0
    _products(dev, A, D, 15)
    A.set_values(L.val)
    assert A.dict_state() == (0, 0, 0)
    n = 2 ** 18 + 64
    rowptr, col, val, _, _ = band(n, np.tile(np.arange(1.0, 6.0), (n, 1)), (-64, -1, 0, 1, 64))
    A = hip.Matrix(dev, rowptr, col, val, nrows=n, ncols=n, fmt=hip.FMT_STENCIL)
    assert A.info()["format"] == hip.FMT_STENCIL and A.dict_state() == (0, 0, 0)
    torch = pytest.importorskip("torch")
    nnz = L.val.size
    ident = hip.Matrix(dev, np.arange(nnz + 1), np.arange(nnz), np.ones(nnz), ncols=nnz, fmt=hip.FMT_CSR)
    dv, change = dev.to_device(2.0 * L.val), torch.cuda.CUDAGraph()
    stream = torch.cuda.ExternalStream(hip.lib().gip_stream(dev.ctx))
    with torch.cuda.graph(change, stream=stream, capture_error_mode="thread_local"):
        ident.spmv_vals(dv, D)
    D.set_values(L.val)
    assert D.dict_state() == (0, 0, 0)


def test_a_batch_makes_none_for_captured_steps(dev):
    """The operators of a batch whose steps are captured take no dictionary's memory (here about 3.5 bytes a row
    more without the graph, over at least ten operators of 2^19 rows and more)."""
    torch = pytest.importorskip("torch")
    from gip_amd import batch

    cavs = [cavity.generate(64, gamma=1e-2) for _ in range(4)]
    used = []
    for graph in (False, True, False, True):
        dev.sync()
        free = torch.cuda.mem_get_info()[0]
        b = batch.Batch(dev, cavs, [1e-2] * 4, pcg_tol=1e-6, use_graph=graph)
        used.append(free - torch.cuda.mem_get_info()[0])
        b.close()
        for _ in range(40):  # the driver may count freed memory a little later
            if free - torch.cuda.mem_get_info()[0] < 4 << 20:
                break
            time.sleep(0.05)
    print(f"[batch memory] without and with a graph {used}", flush=True)
    assert min(used[0::2]) - max(used[1::2]) > 10 * 3 * 2 ** 19


@pytest.mark.parametrize("slots", [2, 7])
@pytest.mark.parametrize("m", [2 ** 17 + 32, 2 ** 17 + 37])
def test_more_rows_than_columns(dev, m, slots):
    """Twice as many rows as columns: a row past the vector's end has no operand of its own."""
    n, rng = 2 * m, np.random.default_rng(16)
    r = np.arange(n)
    col = (r % m)[:, None] + np.arange(slots)[None, :]
    inside = col < m
    rowptr = np.concatenate([[0], np.cumsum(inside.sum(1))])
    val = np.broadcast_to(rng.standard_normal(slots), (n, slots))[inside]
    A = hip.Matrix(dev, rowptr, col[inside], val, nrows=n, ncols=m, fmt=hip.FMT_STENCIL, fp32=True)
    C = hip.Matrix(dev, rowptr, col[inside], val, nrows=n, ncols=m, fmt=hip.FMT_CSR, fp32=True)
    assert A.cols_needed == m and A.info()["format"] == hip.FMT_STENCIL and A.dict_state()[0] != 0
    _products(dev, A, C, 17, fp32=True)

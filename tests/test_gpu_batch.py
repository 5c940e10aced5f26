"""Batched cavities (include/gip_batch.h) against the oracle run instance by
instance on the same operators.

Bar: with the FP64 solver every instance's per-step time, dt, massr and
u, v, w, p fields agree with the oracle to 1e-10 relative (only reduction
orders differ) and PCG iteration counts to +-1; graph replay equals eager
execution bitwise; the mixed-precision batch matches the FP64 oracle to the
solver tolerance.
"""
import time

import numpy as np
import pytest

from gip_amd import batch, cavity, hip
from oracle import pyoracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    d = hip.Device(0)
    yield d
    d.close()


def _cases(tmp_path_factory, sizes, gammas):
    cavs, dirs = [], []
    for k, (n, g) in enumerate(zip(sizes, gammas)):
        c = cavity.generate(n, gamma=g)
        d = tmp_path_factory.mktemp(f"b{k}")
        c.write(d, f"c{k}")
        cavs.append(c)
        dirs.append(d)
    return cavs, dirs


SIZES = [9, 12, 7, 16]
GAMMAS = [1e-2, 1 / 400, 1 / 3200, 1e-3]


def _rel(a, b):
    return abs(a - b) / abs(b) if b else abs(a)


# massr = ||Mres mf||_inf = dt ||L0 p - rhs||_inf (L0: L without the pin) is
# dt |pin p_0| plus the solver residual; on these small cases it is often at
# round-off level (1e-17), where only an absolute comparison is meaningful.
MASSR_FLOOR = 1e-14


def _massr_close(g, w, rel):
    return abs(g - w) <= rel * abs(w) + MASSR_FLOOR


@pytest.mark.parametrize("graph", [False, True])
def test_batch_fp64_matches_oracle_per_instance(dev, tmp_path_factory, graph):
    cavs, dirs = _cases(tmp_path_factory, SIZES, GAMMAS)
    b = batch.Batch(dev, cavs, GAMMAS, pcg_tol=1e-9, pcg_maxit=2000, precision=hip.PCG_FP64, poll=8,
                    use_graph=graph)
    orcs = [pyoracle.Dns(d, f"c{k}", gamma=g, pcg_maxit=2000, pcg_tol=1e-9) for k, (d, g) in
            enumerate(zip(dirs, GAMMAS))]
    same = [True] * len(orcs)
    for step in range(5):
        b.step()
        for k, o in enumerate(orcs):
            w = o.step()
            g = b.info(k)
            print(f"[batch step {step + 1} inst {k}] massr {g['massr']:.6e}/{w['massr']:.6e} "
                  f"pcg {g['pcg_iters']}/{w['pcg_iters']}", flush=True)
            assert g["pcg_status"] == 0
            assert abs(g["pcg_iters"] - w["pcg_iters"]) <= 1
            if same[k]:  # time and dt to 1e-10 while the solves stop at the same iteration
                for key in ("time", "dt"):
                    assert _rel(g[key], w[key]) <= 1e-10, (step, k, key, g[key], w[key])
                assert _massr_close(g["massr"], w["massr"], 1e-4), (step, k, g["massr"], w["massr"])
            same[k] = same[k] and g["pcg_iters"] == w["pcg_iters"]
    for k, o in enumerate(orcs):
        for f in ("u", "v", "w", "p"):
            a, r = b.field(k, f), o.field(f)
            err = np.linalg.norm(a - r) / np.linalg.norm(r)
            assert err <= 1e-7, (k, f, err)


def test_batch_fixed_iterations_match_oracle_to_1e10(dev, tmp_path_factory):
    """With the reference's fixed 100 PCG iterations the batch agrees with the
    oracle per instance to 1e-10 (step numbers and fields)."""
    cavs, dirs = _cases(tmp_path_factory, SIZES, GAMMAS)
    b = batch.Batch(dev, cavs, GAMMAS, pcg_tol=1e-300, pcg_maxit=100, precision=hip.PCG_FP64, poll=10,
                    use_graph=True)
    orcs = [pyoracle.Dns(d, f"c{k}", gamma=g) for k, (d, g) in enumerate(zip(dirs, GAMMAS))]
    for step in range(4):
        b.step()
        for k, o in enumerate(orcs):
            w, g = o.step(), b.info(k)
            assert g["pcg_iters"] == w["pcg_iters"] == 100
            for key in ("time", "dt"):
                assert _rel(g[key], w[key]) <= 1e-10, (step, k, key, g[key], w[key])
            assert _massr_close(g["massr"], w["massr"], 1e-10), (step, k, g["massr"], w["massr"])
    for k, o in enumerate(orcs):
        for f in ("u", "v", "w", "p", "mf"):
            a, r = b.field(k, f), o.field(f)
            assert np.linalg.norm(a - r) <= 1e-10 * np.linalg.norm(r), (k, f)


def test_batch_graph_replay_equals_eager(dev, tmp_path_factory):
    cavs, _ = _cases(tmp_path_factory, SIZES, GAMMAS)
    runs = []
    for graph in (False, True):
        b = batch.Batch(dev, cavs, GAMMAS, pcg_tol=1e-8, precision=hip.PCG_MIXED, poll=4, use_graph=graph)
        out = []
        for _ in range(4):
            t0 = time.perf_counter()
            b.step()
            wall_ms = 1e3 * (time.perf_counter() - t0)
            ph = b.phase_ms()
            print(f"[batch graph={graph}] phases {ph} ms, step wall {wall_ms:.2f} ms", flush=True)
            assert all(v > 0.0 for v in ph.values())
            assert sum(ph.values()) <= wall_ms  # the events bracket device work inside the step
            dev.sync()
            out.append([b.info(k) for k in range(len(cavs))])
        runs.append((out, [b.field(k, "p") for k in range(len(cavs))]))
        b.close()
    assert runs[0][0] == runs[1][0]
    for a, c in zip(runs[0][1], runs[1][1]):
        assert np.array_equal(a, c)


def test_batch_mixed_precision_close_to_fp64_oracle(dev, tmp_path_factory):
    cavs, dirs = _cases(tmp_path_factory, SIZES, GAMMAS)
    b = batch.Batch(dev, cavs, GAMMAS, pcg_tol=1e-10, pcg_maxit=5000, precision=hip.PCG_MIXED, poll=16,
                    autotune=True)
    orcs = [pyoracle.Dns(d, f"c{k}", gamma=g, pcg_maxit=5000, pcg_tol=1e-10) for k, (d, g) in
            enumerate(zip(dirs, GAMMAS))]
    for _ in range(5):
        b.step()
        for k, o in enumerate(orcs):
            w = o.step()
            g = b.info(k)
            assert g["pcg_status"] == 0
            # massr here is the solvers' own residual (round-off level): the
            # mixed run keeps mass as well as the FP64 run, not bit for bit
            assert g["massr"] <= max(100 * w["massr"], 1e-12), (k, g["massr"], w["massr"])
    for k, o in enumerate(orcs):
        for f in ("u", "v", "w", "p"):
            a, r = b.field(k, f), o.field(f)
            err = np.linalg.norm(a - r) / np.linalg.norm(r)
            print(f"[batch mixed inst {k} {f}] rel {err:.2e}")
            assert err <= 1e-7, (k, f, err)
    print("[batch layouts]", b.layouts())


def test_batch_single_instance_on_c100k_matches_oracle(dev, c100k_root):
    """The shipped C100K case (tetrahedral cells, merged to one partition) as
    a one-instance batch: the device-resident, graph-captured step against
    the oracle with the reference's fixed 100 PCG iterations, to 1e-10."""
    cav = cavity.read(c100k_root, "C100K")
    b = batch.Batch(dev, [cav], [1e-3], pcg_tol=1e-300, pcg_maxit=100, precision=hip.PCG_FP64, poll=100,
                    use_graph=True)
    orc = pyoracle.Dns(c100k_root, "C100K", gamma=1e-3)
    for step in range(3):
        b.step()
        w, g = orc.step(), b.info(0)
        print(f"[C100K batch step {step + 1}] massr {g['massr']:.9e} dt {g['dt']:.9e} | oracle {w['massr']:.9e}",
              flush=True)
        assert g["pcg_iters"] == w["pcg_iters"] == 100
        for key in ("time", "dt"):
            assert _rel(g[key], w[key]) <= 1e-10, (step, key, g[key], w[key])
        assert _massr_close(g["massr"], w["massr"], 1e-10), (step, g["massr"], w["massr"])
    for f in ("u", "v", "w", "p", "mf"):
        a, r = b.field(0, f), orc.field(f)
        assert np.linalg.norm(a - r) <= 1e-10 * np.linalg.norm(r), f
    b.close()


def test_batch_argument_errors(dev):
    """gip_batch_create rejects a non-positive tolerance and a cavity that
    lacks the integrator's operators."""
    full = cavity.generate(8, gamma=1e-2)
    with pytest.raises(hip.HipError) as e:
        batch.Batch(dev, [full], [1e-2], pcg_tol=0.0)
    assert e.value.code == hip.EINVAL
    lap_only = cavity.generate(8, gamma=1e-2, ops=cavity.OP_BITS["L"])
    with pytest.raises(hip.HipError) as e:
        batch.Batch(dev, [full, lap_only], [1e-2, 1e-2], pcg_tol=1e-8)
    assert e.value.code == hip.EINVAL


# One, two or four chunks per workgroup of the sweeps by the size of the
# batch, partial units at an instance's end, and an instance of more than
# 2048 chunks (81^3), with which one-workgroup kernels form the scalars: an
# instance gives what it gives alone.  40 iterations without a tolerance, so
# only the order of the sums differs: FP64 40 x 2 steps x 1e-16 and its
# growth through the iteration, bounded by 1e-9; in mixed precision a flipped
# rounding of alpha or beta to FP32 (6e-8) in each of 80 iterations, 1e-5.
@pytest.mark.parametrize("precision,bound", [(hip.PCG_FP64, 1e-9), (hip.PCG_MIXED, 1e-5)])
@pytest.mark.parametrize("sizes", [[20, 57, 57, 57], [20, 64, 64, 64, 64, 9], [20, 81, 9]])
def test_instance_in_a_large_batch_is_the_instance_alone(dev, sizes, precision, bound):
    def run(ns, poll):
        cavs = [cavity.generate(n, gamma=1e-2) for n in ns]
        b = batch.Batch(dev, cavs, [1e-2] * len(ns), pcg_tol=1e-30, pcg_maxit=40, precision=precision, poll=poll,
                        use_graph=False)
        for _ in range(2):
            b.step()
        out = [(b.info(k)["pcg_iters"], b.field(k, "p")) for k in range(len(ns))]
        b.close()
        return out

    got = run(sizes, 7)
    for k in (0, len(sizes) - 2, len(sizes) - 1):
        (iters, p), = run([sizes[k]], 7)
        assert got[k][0] == iters
        assert np.abs(got[k][1] - p).max() <= bound * np.abs(p).max(), sizes[k]


# A breakdown is decided inside the update sweep, by every workgroup of the
# instance from the same sums: the broken instance keeps the pressure it had
# (its start, zero; in mixed precision after the coarse step, here below
# 1e-20), in every chunk, and its neighbours advance as if it were whole.  Its
# p.Ap overflows on a finite direction, 1e300 r (FP32: 1e20 r).
@pytest.mark.parametrize("precision,diag,off", [(hip.PCG_FP64, 1e-300, 1e100), (hip.PCG_MIXED, 1e-20, 1e25)])
@pytest.mark.parametrize("sizes", [[12, 20, 9], [20, 57, 9], [33, 72, 64, 64]])
def test_a_breakdown_leaves_the_instance_and_its_neighbours_alone(dev, sizes, precision, diag, off):
    def run(broken):
        cavs = [cavity.generate(n, gamma=1e-2) for n in sizes]
        if broken:
            L = cavs[1].op("L")
            row = np.repeat(np.arange(L.nrows), np.diff(L.rowptr))
            L.val[:] = np.where(L.col == row, diag, off)
        b = batch.Batch(dev, cavs, [1e-2] * len(sizes), pcg_tol=1e-8, pcg_maxit=60, precision=precision)
        b.step()
        out = [(b.info(k), b.field(k, "p")) for k in range(len(sizes))]
        b.close()
        return out

    whole, got = run(False), run(True)
    info, p = got[1]
    n = info["n_inner"]
    print(f"[batch breakdown {sizes}] iters {info['pcg_iters']} status {info['pcg_status']}", flush=True)
    assert info["pcg_status"] == hip.EBREAKDOWN and info["pcg_iters"] == 0
    assert np.abs(p[:n]).max() <= (0.0 if precision == hip.PCG_FP64 else 1e-20)
    for k in [0] + list(range(2, len(sizes))):
        assert got[k][0]["pcg_iters"] == whole[k][0]["pcg_iters"] > 0
        assert np.array_equal(got[k][1], whole[k][1])

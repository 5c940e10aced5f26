"""Performance cases of gip_amd: what a program built on it has it do.

A case is one call (or one short run of calls) through the public Python
entry points: a vector reduction, an operator product, a pressure solve in
FP64 or mixed precision, time steps of the integrator, a step of a batch of
cavities, a gradient.  Sizes are those of the repository's own
configurations and tests (46^3, 64^3, 97^3, 128^3 clustered, 256^3) and the
ranges around them.

Operators come from the cavity generator (uniform and tanh-clustered meshes,
odd and ragged sides), or from it with the cells renumbered irregularly (what
an unstructured mesh gives: no shared column offsets).  Vectors and fields
are made from the seed on the device.
"""
import functools
import math

import numpy as np
import torch

from gip_amd import adjoint, batch, cavity, dns, hip

GAMMA = 1e-2  # 1/Re of the generated cases


def listed():
    return [
        # a dot product of the host-driven solver sequence at the shipped case's size: launch and return latency
        {"name": "dot_46", "kind": "dot", "n": 46 ** 3},
        # one operator product at the same size (every phase of a small step is made of these)
        {"name": "spmv_46", "kind": "spmv", "nx": 46, "ny": 46, "nz": 46, "beta": 0.0, "fp32": False, "scatter": False},
        # the product of the largest configuration
        {"name": "spmv_256", "kind": "spmv", "nx": 256, "ny": 256, "nz": 256, "beta": 0.0, "fp32": False,
         "scatter": False},
        # the pressure solve of a time step as the reference runs it: 100 fixed iterations, a small mesh
        {"name": "pcg_fixed_46", "kind": "pcg", "nx": 46, "ny": 46, "nz": 46, "beta": 0.0, "mixed": False,
         "maxit": 100, "tol": 0.0, "scatter": False},
        # the same on an irregularly numbered mesh (sliced ELL instead of the stencil layout)
        {"name": "pcg_fixed_irregular_60", "kind": "pcg", "nx": 60, "ny": 60, "nz": 60, "beta": 0.0, "mixed": False,
         "maxit": 100, "tol": 0.0, "scatter": True},
        # the wall-clustered 128^3 configuration solved to convergence in FP64
        {"name": "pcg_clustered_128", "kind": "pcg", "nx": 128, "ny": 128, "nz": 128, "beta": 1.5, "mixed": False,
         "maxit": 4000, "tol": 1e-10, "scatter": False},
        # the largest configuration with the reference's fixed iteration count
        {"name": "pcg_fixed_256", "kind": "pcg", "nx": 256, "ny": 256, "nz": 256, "beta": 0.0, "mixed": False,
         "maxit": 100, "tol": 0.0, "scatter": False},
        # mixed precision, an odd side: slices that straddle the mesh lines
        {"name": "pcg_mixed_97", "kind": "pcg", "nx": 97, "ny": 97, "nz": 97, "beta": 0.0, "mixed": True,
         "maxit": 4000, "tol": 1e-12, "scatter": False},
        # mixed precision at the largest configuration: the headline solve, to the residual at which the pressure
        # itself (1e3 times the residual's error here) agrees with an FP64 solve to 1e-9
        {"name": "pcg_mixed_256", "kind": "pcg", "nx": 256, "ny": 256, "nz": 256, "beta": 0.0, "mixed": True,
         "maxit": 6000, "tol": 1e-12, "scatter": False},
        # time steps of a small cavity with the device solver, fields read at the end
        {"name": "steps_46", "kind": "steps", "n": 46, "beta": 0.0, "mode": "fused", "maxit": 100, "tol": 0.0,
         "steps": 4},
        # uneven cavities advanced together, mixed precision
        {"name": "batch_12", "kind": "batch", "count": 12, "low": 32, "high": 72, "mixed": True, "tol": 1e-11,
         "steps": 1},
        # a gradient through a few steps: forward run, checkpoints, reverse run
        {"name": "gradient_32", "kind": "gradient", "n": 32, "steps": 4, "every": 2},
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _sides(rng, low, high):
    """Three sides: equal half of the time, else each within a quarter of the first."""
    n = _log(rng, low, high)
    if rng.random() < 0.5:
        return {"nx": n, "ny": n, "nz": n}
    return {"nx": n, "ny": min(high, max(low, int(n * rng.uniform(0.75, 1.25)))),
            "nz": min(high, max(low, int(n * rng.uniform(0.75, 1.25))))}


def draw(rng):
    kind = rng.choice(["dot", "spmv", "spmv", "pcg_fixed", "pcg_fixed", "pcg_tol", "pcg_mixed", "pcg_mixed", "steps",
                       "batch", "gradient"])
    beta = rng.choice([0.0, 0.0, round(rng.uniform(1.0, 2.0), 3)])
    if kind == "dot":
        return {"kind": "dot", "n": _log(rng, 4000, 256 ** 3)}
    if kind == "spmv":
        scatter = rng.random() < 0.25
        return {"kind": "spmv", **_sides(rng, 24, 96 if scatter else 224), "beta": beta, "fp32": rng.random() < 0.5,
                "scatter": scatter}
    if kind == "pcg_fixed":
        scatter = rng.random() < 0.25
        return {"kind": "pcg", **_sides(rng, 24, 96 if scatter else 224), "beta": beta, "mixed": False,
                "maxit": _log(rng, 20, 200), "tol": 0.0, "scatter": scatter}
    if kind == "pcg_tol":
        return {"kind": "pcg", **_sides(rng, 24, 136), "beta": beta, "mixed": False, "maxit": 6000, "tol": 1e-10,
                "scatter": False}
    if kind == "pcg_mixed":
        return {"kind": "pcg", **_sides(rng, 24, 176), "beta": beta, "mixed": True, "maxit": 6000, "tol": 1e-12,
                "scatter": False}
    if kind == "steps":
        mode = rng.choice(["reference", "fused", "mixed"])
        return {"kind": "steps", "n": _log(rng, 20, 64), "beta": beta, "mode": mode,
                "maxit": 4000 if mode == "mixed" else 100, "tol": 1e-12 if mode == "mixed" else 0.0,
                "steps": rng.randint(1, 3)}
    if kind == "batch":
        low = rng.randint(16, 40)
        return {"kind": "batch", "count": rng.randint(2, 10), "low": low, "high": low + rng.randint(0, 24),
                "mixed": rng.random() < 0.7, "tol": 1e-11, "steps": 1}
    return {"kind": "gradient", "n": _log(rng, 16, 40), "steps": rng.randint(2, 5), "every": rng.randint(1, 3)}


# ---- inputs -----------------------------------------------------------------


@functools.lru_cache(maxsize=1)
def _device():
    return hip.Device(0)


class _Raw:
    """A device array of the library as torch sees device memory."""

    def __init__(self, a):
        self.owner = a
        self.__cuda_array_interface__ = {"shape": (a.n,), "typestr": a.dtype.str, "data": (a.ptr.value, False),
                                         "version": 2}


def _tensor(a):
    return torch.as_tensor(_Raw(a), device="cuda")


def _fill(a, t):
    """A library array holding the values of a torch tensor."""
    _tensor(a).copy_(t)
    return a


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


@functools.lru_cache(maxsize=3)
def _laplacian(nx, ny, nz, beta, scatter):
    """The pressure Laplacian as host CSR arrays (rowptr, col, val, cells, vector length)."""
    cav = cavity.generate(nx, ny, nz, beta=beta, gamma=GAMMA, ops=cavity.OP_BITS["L"])
    a, n = cav.op("L"), cav.n_inner
    rowptr, col, val = a.rowptr.copy(), a.col.copy(), a.val.copy()
    if scatter:
        # cells renumbered at random inside windows of about 2000, columns ascending in each row
        rng = np.random.RandomState(n % 1000003)
        new = np.argsort(np.arange(n) // 2000 + rng.random_sample(n) * 0.999, kind="stable").argsort().astype(np.int32)
        row = np.repeat(new, np.diff(rowptr))
        to = np.concatenate([new, np.arange(n, max(cav.n_all, n), dtype=np.int32)])
        col = to[col]
        order = np.lexsort((col, row))
        col, val = np.ascontiguousarray(col[order]), np.ascontiguousarray(val[order])
        rowptr = np.concatenate([[0], np.cumsum(np.bincount(row, minlength=n))]).astype(np.int32)
    return rowptr, col, val, n, cav.n_all


def _lap(case):
    return _laplacian(case["nx"], case["ny"], case["nz"], case["beta"], case["scatter"])


def _pressure(case, seed):
    """A pressure-like field on the cells: a few smooth modes with small noise, zero mean, zero on the ghosts."""
    _, _, _, n, n_all = _lap(case)
    g = _generator(seed)
    axes = [(torch.arange(m, device="cuda", dtype=torch.float64) + 0.5) / m for m in (case["nx"], case["ny"], case["nz"])]
    field = 0.02 * torch.randn(case["nz"], case["ny"], case["nx"], generator=g, device="cuda", dtype=torch.float64)
    for c, kx, ky, kz in zip(torch.randn(6, generator=g, device="cuda", dtype=torch.float64),
                             *torch.randint(0, 6, (3, 6), generator=g, device="cuda")):
        mode = [torch.cos(math.pi * k * x) for k, x in zip((kx, ky, kz), axes)]
        field += c * mode[2][:, None, None] * mode[1][None, :, None] * mode[0][None, None, :]
    x = torch.zeros(n_all, device="cuda", dtype=torch.float64)
    x[:n] = (field - field.mean()).reshape(-1)
    return x


def _velocity(n, seed, k):
    g = _generator(1000 * int(seed) + k)
    s = (torch.arange(n, device="cuda", dtype=torch.float64) + 0.5) / n
    bump = torch.sin(math.pi * s)
    field = bump[:, None, None] * bump[None, :, None] * bump[None, None, :]
    amp = 1.0 + 0.2 * torch.randn(n, n, n, generator=g, device="cuda", dtype=torch.float64)
    return (0.1 * field * amp).reshape(-1).cpu().numpy()


def prepare(case, seed):
    dev = _device()
    kind = case["kind"]
    if kind == "dot":
        g = _generator(seed)
        v = [_fill(dev.array(case["n"]), torch.randn(case["n"], generator=g, device="cuda", dtype=torch.float64) + 0.25)
             for _ in range(2)]
        state = {"x": v[0], "y": v[1]}
    elif kind == "spmv":
        rowptr, col, val, n, n_all = _lap(case)
        dt = np.float32 if case["fp32"] else np.float64
        y = dev.array(n, dt)
        state = {"A": hip.Matrix(dev, rowptr, col, val, nrows=n, ncols=n_all, fp32=case["fp32"]), "y": y,
                 "x": _fill(dev.array(n_all, dt), _pressure(case, seed)), "out": _tensor(y)}
    elif kind == "pcg":
        rowptr, col, val, n, n_all = _lap(case)
        A = hip.Matrix(dev, rowptr, col, val, nrows=n, ncols=n_all, fp32=case["mixed"])
        # the right-hand side of a known pressure
        b, zero, x = dev.array(n_all), _fill(dev.array(n_all), torch.zeros(n_all, device="cuda")), dev.array(n_all)
        _tensor(b).zero_()
        _fill(x, _pressure(case, seed))
        torch.cuda.synchronize()
        A.spmv(x, b)
        state = {"A": A, "solver": hip.PCG(A, n_all), "b": b, "x": x, "x0": zero, "out": _tensor(x)}
    elif kind == "steps":
        cav = _cavity(case["n"], case["beta"])
        sim = dns.Simulation(cavity=cav, gamma=GAMMA, pcg_maxit=case["maxit"], pcg_tol=case["tol"],
                             pcg_mode=case["mode"])
        for k, f in enumerate("uvw"):
            v = sim.field(f)
            v[:cav.n_inner] = _velocity(case["n"], seed, k)
            sim.set_field(f, v)
        state = {"sim": sim}
    elif kind == "batch":
        span = max(1, case["count"] - 1)
        sides = [case["low"] + (case["high"] - case["low"]) * i // span for i in range(case["count"])]
        rng = np.random.RandomState(int(seed) % (1 << 31))
        state = {"batch": batch.Batch(dev, [_cavity(n, 0.0) for n in sides],
                                      [float(10 ** -rng.uniform(2.0, 3.5)) for _ in sides], pcg_tol=case["tol"],
                                      precision=hip.PCG_MIXED if case["mixed"] else hip.PCG_FP64),
                 "count": case["count"]}
    else:
        cav = _cavity(case["n"], 0.0)
        n = case["n"]
        s = (np.arange(n) + 0.5) / n
        lid = np.outer(np.sin(np.pi * s), np.sin(np.pi * s)).ravel()
        lid = lid * (1.0 + 0.1 * np.random.RandomState(int(seed) % (1 << 31)).standard_normal(lid.size))
        state = {"adjoint": adjoint.Adjoint(dev, cav, steps=case["steps"], checkpoint_every=case["every"], gamma=GAMMA),
                 "lid": lid, "start": [_velocity(n, seed, k) for k in range(3)]}
    torch.cuda.synchronize()
    return {"case": dict(case), **state}


@functools.lru_cache(maxsize=24)
def _cavity(n, beta):
    return cavity.generate(n, beta=beta, gamma=GAMMA)


# ---- one pass ---------------------------------------------------------------


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "dot":
        return hip.dot(state["x"], state["y"])
    if kind == "spmv":
        (state["A"].spmv32 if case["fp32"] else state["A"].spmv)(state["x"], state["y"])
        return state["out"]
    if kind == "pcg":
        state["solver"].solve(state["b"], state["x"], state["x0"], maxit=case["maxit"], tol=case["tol"],
                              precision=hip.PCG_MIXED if case["mixed"] else hip.PCG_FP64)
        return state["out"]
    if kind == "steps":
        sim = state["sim"]
        for _ in range(case["steps"]):
            info = sim.step()
        return {**{f: sim.field(f) for f in ("u", "v", "w", "p", "mf")}, "time": info["time"], "dt": info["dt"]}
    if kind == "batch":
        b = state["batch"]
        for _ in range(case["steps"]):
            b.step()
        return [{**{f: b.field(i, f) for f in ("u", "p", "mf")}, "dt": b.info(i)["dt"]} for i in range(state["count"])]
    a = state["adjoint"]
    objective = a.forward(state["lid"], *state["start"])
    return {"objective": objective, "gradient": list(a.backward())}


# ---- what a pass cannot do without ------------------------------------------


def _iterations(case):
    """Iterations of a solve: the fixed count, or about what a zero-mean right-hand side of this mesh takes."""
    if not case["tol"] > 0.0:
        return case["maxit"]
    longest = max(case["nx"], case["ny"], case["nz"])
    return int(longest * (6.5 if case["mixed"] else 10.5) * (1.3 if case["beta"] else 1.0))


def work(case):
    """Bytes and operations of a pass: operator values and vectors once per product or iteration."""
    kind = case["kind"]
    if kind == "dot":
        return {"bytes": 16.0 * case["n"], "flops": 2.0 * case["n"]}
    if kind in ("spmv", "pcg"):
        n = float(case["nx"] * case["ny"] * case["nz"])
        nnz = 7.0 * n
        if kind == "spmv":
            w = 4 if case["fp32"] else 8
            return {"bytes": w * (nnz + 2 * n), "flops": 2 * nnz}
        w, it = (4 if case["mixed"] else 8), _iterations(case)
        # per iteration: the operator and the preconditioner read; x, r and p read and written
        return {"bytes": it * w * (nnz + 7 * n), "flops": it * (2 * nnz + 11 * n)}
    if kind == "steps":
        n = float(case["n"] ** 3)
        it = case["maxit"] if not case["tol"] > 0.0 else 5 * case["n"]
        one = 8 * (13 * n + 100 * n) + it * (4 if case["mode"] == "mixed" else 8) * 14 * n
        return {"bytes": case["steps"] * one, "flops": case["steps"] * n * (25 * it + 200)}
    if kind == "batch":
        span = max(1, case["count"] - 1)
        sides = [case["low"] + (case["high"] - case["low"]) * i // span for i in range(case["count"])]
        one = sum(n ** 3 * (904 + 5 * n * (4 if case["mixed"] else 8) * 14) for n in sides)
        return {"bytes": float(case["steps"] * one), "flops": float(case["steps"] * sum(n ** 3 * 125 * n for n in sides))}
    n = float(case["n"] ** 3)
    # forward, recomputed forward and reverse: a solve of about 9 iterations per cell of a side in each
    one = 3 * (904 * n + 9 * case["n"] * 8 * 14 * n)
    return {"bytes": case["steps"] * one, "flops": case["steps"] * 3 * n * (25 * 9 * case["n"] + 200)}


# ---- the same in plain 64-bit torch -----------------------------------------


def exact(case, seed):
    """FP64 results by plain torch: the dot product, the product with the CSR arrays, the pressure behind the
    right-hand side of a converged solve, the iterate of a fixed number of Jacobi-CG iterations; None otherwise."""
    kind = case["kind"]
    if kind == "dot":
        g = _generator(seed)
        x, y = (torch.randn(case["n"], generator=g, device="cuda", dtype=torch.float64) + 0.25 for _ in range(2))
        return torch.dot(x, y)
    if kind not in ("spmv", "pcg"):
        return None
    rowptr, col, val, n, n_all = _lap(case)
    x = _pressure(case, seed)
    if kind == "pcg" and case["tol"] > 0.0:
        return x
    A = torch.sparse_csr_tensor(torch.from_numpy(rowptr).cuda(), torch.from_numpy(col).cuda(),
                                torch.from_numpy(val).cuda(), size=(n, n_all))
    if kind == "spmv":
        return A @ (x.float().double() if case["fp32"] else x)
    rows = np.repeat(np.arange(n, dtype=np.int32), np.diff(rowptr))
    diag = torch.from_numpy(val[col == rows]).cuda()
    b = A @ x
    # Jacobi-CG from zero; the ghosts stay zero
    full = torch.zeros(n_all, device="cuda", dtype=torch.float64)
    z, r = torch.zeros_like(b), b.clone()
    s = r / diag
    p, rho = s.clone(), torch.dot(r, s)
    for _ in range(case["maxit"]):
        full[:n] = p
        q = A @ full
        alpha = rho / torch.dot(p, q)
        z += alpha * p
        r -= alpha * q
        s = r / diag
        new = torch.dot(r, s)
        p = s + (new / rho) * p
        rho = new
    full[:n] = z
    return full

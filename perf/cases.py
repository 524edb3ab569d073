"""Workloads of the solve path, as programs call it through the Python surface.

A case names an operation, a graph and its size. The host factorization of a
graph (``apxchol_amd.factorize``) is computed once per process; every
preparation builds its own ``Solver`` (or ``Group``) on it, uploads it and
draws the right-hand sides from its seed.

operations  solve        Solver.solve on device vectors (one right-hand side)
            solve_host   Solver.solve on host vectors (copies included)
            solve_batch  Solver.solve_batch, k right-hand sides in one block
            apply        Solver.apply, one preconditioner application
            apply_batch  Solver.apply_batch, k columns at once
            spmv         Solver.spmv
            group        Group.solve over k small 2-D grids, one launch a step
graphs      grid2d / grid3d (unit weights), sddm3d (lognormal weights and a
            diagonal excess), aniso3d (axis weights 1 / 10 / 100, lognormal),
            rmat (power law, edge factor 16); size is the side or the scale
precision   vector width of the triangular sweeps ("fp64" is the default of
            the Solver, "fp32" the mixed configuration)
"""
from functools import lru_cache

import numpy as np
import torch

import apxchol_amd as ax
from apxchol_amd import matgen as mg

TOL = 1e-8


def listed():
    def case(name, op, graph, size, precision, k=1):
        return {"name": name, "op": op, "graph": graph, "size": size, "precision": precision, "k": k}
    return [
        # The smallest resident factor of the serving mix: launches and latency.
        case("solve grid2d 100 mixed", "solve", "grid2d", 100, "fp32"),
        # The small 2-D workload with every option at its default.
        case("solve grid2d 256 fp64", "solve", "grid2d", 256, "fp64"),
        # A caller that holds NumPy vectors, on a 3-D factor of the serving mix.
        case("solve_host grid3d 48 fp64", "solve_host", "grid3d", 48, "fp64"),
        # A mid-size SDDM system of odd side in the default precision.
        case("solve sddm3d 89 fp64", "solve", "sddm3d", 89, "fp64"),
        # The benchmark's headline: one mixed solve of the 128^3 SDDM grid.
        case("solve sddm3d 128 mixed", "solve", "sddm3d", 128, "fp32"),
        # Power-law graphs: thousands of dependent levels and hub rows.
        case("solve rmat 14 fp64", "solve", "rmat", 14, "fp64"),
        case("solve rmat 18 mixed", "solve", "rmat", 18, "fp32"),
        # The benchmark's blocked workload.
        case("solve_batch aniso3d 64 k32 mixed", "solve_batch", "aniso3d", 64, "fp32", 32),
        # A few right-hand sides at once, an odd count, default precision.
        case("solve_batch grid3d 48 k5 fp64", "solve_batch", "grid3d", 48, "fp64", 5),
        # The preconditioner alone, inside a caller's own Krylov method.
        case("apply sddm3d 63 fp64", "apply", "sddm3d", 63, "fp64"),
        case("apply_batch grid2d 316 k8 fp64", "apply_batch", "grid2d", 316, "fp64", 8),
        # Many small factors, one right-hand side each.
        case("group 16 grid2d 64 mixed", "group", "grid2d", 64, "fp32", 16),
    ]


# Largest drawn side (or scale) of each graph, per operation class: a blocked
# operation moves k columns, so its sizes end lower.
_RANGE = {"grid2d": (24, 1000, 500), "grid3d": (9, 110, 56), "sddm3d": (9, 112, 56), "aniso3d": (9, 80, 56),
          "rmat": (9, 18, 15)}


def draw(rng):
    op = rng.choice(["solve", "solve", "solve", "solve_host", "solve_batch", "solve_batch", "apply", "apply_batch",
                     "spmv", "group"])
    graph = "grid2d" if op == "group" else rng.choice(["grid2d", "grid3d", "sddm3d", "aniso3d", "rmat"])
    blocked = op in ("solve_batch", "apply_batch")
    lo, hi1, hik = _RANGE[graph]
    hi = 128 if op == "group" else hik if blocked else hi1
    if graph == "rmat":
        size = rng.randint(lo, hi)
    else:
        size = int(round(lo * (hi / lo) ** rng.random()))
    k = rng.randint(2, 32) if blocked else rng.randint(2, 24) if op == "group" else 1
    # Applications return the sweeps' outputs as they are; the mixed
    # configuration exists for solves, whose iteration stays in fp64.
    precision = rng.choice(["fp64", "fp32"]) if op.startswith("solve") or op == "group" else "fp64"
    return {"op": op, "graph": graph, "size": size, "precision": precision, "k": k}


@lru_cache(maxsize=None)
def _system(graph, size, index=0):
    """(A, factor, component labels or None) of a graph; index varies the
    sizes of a group's members a little, as separate small systems differ."""
    A, _ = mg.workload(f"{graph}_{size + index % 5}")
    F = ax.factorize(A, seed=0)
    labels = None
    if not F.sddm:
        import scipy.sparse.csgraph as csg
        labels = csg.connected_components(A, directed=False)[1]
    return A, F, labels


def _rhs(system, rng):
    """A N(0,1) right-hand side, projected onto the range of a Laplacian."""
    A, _, labels = system
    b = rng.standard_normal(A.shape[0])
    if labels is not None:
        count = np.bincount(labels)
        b -= (np.bincount(labels, weights=b) / count)[labels]
        b[count[labels] == 1] = 0.0
    return b


def _inputs(case, seed):
    """The systems and host right-hand sides of a case."""
    rng = np.random.default_rng([seed, 17])
    if case["op"] == "group":
        systems = [_system(case["graph"], case["size"], i) for i in range(case["k"])]
        return systems, [_rhs(s, rng) for s in systems]
    system = _system(case["graph"], case["size"])
    return [system], [_rhs(system, rng) for _ in range(case["k"])]


def prepare(case, seed):
    systems, bs = _inputs(case, seed)
    op = case["op"]
    solvers = [ax.Solver(A, factor=F, precision=case["precision"], tol=TOL) for A, F, _ in systems]
    state = {"op": op, "solver": solvers[0]}
    if op == "group":
        state["solver"] = ax.Group(solvers)
        state["b"] = [torch.tensor(b, device="cuda") for b in bs]
    elif op == "solve_host":
        state["b"] = bs[0]
    elif op in ("solve_batch", "apply_batch"):
        state["b"] = torch.tensor(np.stack(bs), device="cuda")
    else:
        state["b"] = torch.tensor(bs[0], device="cuda")
    return state


def run(state):
    s, b, op = state["solver"], state["b"], state["op"]
    if op in ("solve", "solve_host"):
        r = s.solve(b)
        return {"x": r.x, "iterations": r.iterations}
    if op == "solve_batch":
        x, rs = s.solve_batch(b)
        return {"x": x, "iterations": [r.iterations for r in rs]}
    if op == "group":
        x, rs = s.solve(b)
        return {"x": x, "iterations": [r.iterations for r in rs]}
    if op == "spmv":
        return {"y": s.spmv(b)}
    # A Krylov method's first application (the centring schedule counts them).
    s.reset_apply_count()
    return {"z": s.apply(b) if op == "apply" else s.apply_batch(b)}


def _sizes(case):
    """(rows, operator entries, factor off-diagonals), the last two by the
    graphs' mean row lengths."""
    graph, size = case["graph"], case["size"]
    if graph == "rmat":
        n = 1 << size
        return n, 28 * n, 26 * n
    if graph == "grid2d":
        n = size * size
        return n, 5 * n - 4 * size, int(4.4 * n)
    n = size ** 3
    return n, 7 * n - 6 * size * size, int(8.2 * n)


def work(case):
    """One pass over the operator (fp64 values, 32-bit columns) and the two
    sweeps over the factor (fp32 values) per iteration, for k columns; a
    solve to 1e-8 takes about 25 iterations on these graphs."""
    n, nnz, off = _sizes(case)
    k, op = case["k"], case["op"]
    vec = 8 if case["precision"] == "fp64" else 4
    copies = k if op == "group" else 1      # members have operators and factors of their own
    cols = 1 if op == "group" else k
    spmv = {"bytes": 12 * nnz + 4 * n + 16 * n * cols, "flops": 2 * nnz * cols}
    sweeps = {"bytes": 2 * (8 * off + 8 * n) + (8 + 3 * vec) * n * cols, "flops": 4 * off * cols + 2 * n * cols}
    if op == "spmv":
        return spmv
    if op.startswith("apply"):
        return sweeps
    vectors = {"bytes": 88 * n * cols, "flops": 12 * n * cols}
    return {m: 25 * copies * (spmv[m] + sweeps[m] + vectors[m]) for m in ("bytes", "flops")}


def _solve64(system, b):
    """The minimum-norm solution of A x = b to fp64 rounding, by conjugate
    gradients with the diagonal as preconditioner."""
    A, _, labels = system
    S = A.tocsr()
    d = S.diagonal()
    inv = np.where(d > 0, 1.0 / np.where(d > 0, d, 1.0), 0.0)
    x, r = np.zeros_like(b), b.copy()
    z = inv * r
    p, rz, nb = z.copy(), float(r @ z), float(np.linalg.norm(b))
    for _ in range(20000):
        if np.linalg.norm(r) <= 1e-13 * nb:
            break
        q = S @ p
        a = rz / float(p @ q)
        x += a * p
        r -= a * q
        z = inv * r
        rz, old = float(r @ z), rz
        p = z + (rz / old) * p
    return x if labels is None else x - x.mean()


def exact(case, seed):
    """Solutions and products in 64 bits by scipy. An application of the
    randomized preconditioner has no value outside this package, and the
    larger solves take minutes on the host."""
    op = case["op"]
    if op.startswith("apply"):
        return None
    n, nnz, _ = _sizes(case)
    if op != "spmv" and nnz * case["k"] > 6_000_000:
        return None
    systems, bs = _inputs(case, seed)
    if op == "spmv":
        return {"y": torch.from_numpy(systems[0][0] @ bs[0])}
    if case["graph"] == "rmat":
        return None      # constants of small components are free beside the large one
    systems = systems if op == "group" else systems * len(bs)
    x = [_solve64(s, b) for s, b in zip(systems, bs)]
    if op == "group":
        return {"x": [torch.from_numpy(v) for v in x], "iterations": [None] * len(x)}
    if op == "solve_batch":
        return {"x": torch.from_numpy(np.stack(x)), "iterations": [None] * len(x)}
    return {"x": torch.from_numpy(x[0]), "iterations": None}

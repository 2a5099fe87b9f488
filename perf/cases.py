"""The workloads by which this library's speed is judged, as a user's program
runs them: single-system CG and BiCGSTAB solves on device buffers, batched CG
on host buffers, and the set-up of a new matrix with its first product.

Every solve runs to a true relative residual of 1e-12.  At that tolerance the
returned x agrees with the solution to about ten digits whatever the rounding
of the way there, so x is a number that two builds can be compared on.
Right-hand sides are b = A x*, x* uniform in (-1, 1).
"""
import functools
import importlib

import numpy as np
import torch

mf = importlib.import_module("mille-feillue_amd")

TOL = 1e-12
FP32_TAU = 2.0 ** -24  # per-tile rounding that lets every tile be FP32


def listed():
    return [
        # the smallest call: one workgroup, latency alone (a small 2D grid,
        # solved inside an outer loop of the caller)
        {"name": "cg_fp64_laplace2d_30x31", "kind": "cg", "matrix": "laplace2d", "nx": 30, "ny": 31, "nz": 1, "mixed": False, "tau": 0.0},
        # a 2D grid of ordinary size: hundreds of short, dependent iterations
        {"name": "cg_fp64_laplace2d_251x257", "kind": "cg", "matrix": "laplace2d", "nx": 251, "ny": 257, "nz": 1, "mixed": False, "tau": 0.0},
        # a small 3D grid on lossless E4M3 tiles (the default mixed precision)
        {"name": "cg_mixed_poisson3d_33x31x29", "kind": "cg", "matrix": "poisson3d", "nx": 33, "ny": 31, "nz": 29, "mixed": True, "tau": 0.0},
        # an ordinary 3D grid of odd sides, mixed
        {"name": "cg_mixed_poisson3d_83x79x77", "kind": "cg", "matrix": "poisson3d", "nx": 83, "ny": 79, "nz": 77, "mixed": True, "tau": 0.0},
        # the headline system of the benchmark, in FP64 and mixed
        {"name": "cg_fp64_poisson3d_128", "kind": "cg", "matrix": "poisson3d", "nx": 128, "ny": 128, "nz": 128, "mixed": False, "tau": 0.0},
        {"name": "cg_mixed_poisson3d_128", "kind": "cg", "matrix": "poisson3d", "nx": 128, "ny": 128, "nz": 128, "mixed": True, "tau": 0.0},
        # the largest: more rows than registers and LDS hold, mixed
        {"name": "cg_mixed_poisson3d_151x149x147", "kind": "cg", "matrix": "poisson3d", "nx": 151, "ny": 149, "nz": 147, "mixed": True, "tau": 0.0},
        # nonsymmetric 27-point systems: a small one in FP64 ...
        {"name": "bicgstab_fp64_convdiff_39", "kind": "bicgstab", "matrix": "convdiff3d", "nx": 39, "ny": 39, "nz": 39, "mixed": False, "tau": 0.0},
        # ... and the benchmark's size on FP32-rounded tiles
        {"name": "bicgstab_fp32tiles_convdiff_96", "kind": "bicgstab", "matrix": "convdiff3d", "nx": 96, "ny": 96, "nz": 96, "mixed": True, "tau": FP32_TAU},
        # no stencil: random columns, row lengths from 2 to thousands
        {"name": "cg_fp64_random_spd_200001", "kind": "cg", "matrix": "random_spd", "nx": 200001, "ny": 1, "nz": 1, "mixed": False, "tau": 0.0},
        # many systems of uneven size, eight right-hand sides each
        {"name": "batch_48x8_500_to_8000_rows", "kind": "batch", "systems": 48, "nrhs": 8, "least": 500, "most": 8000, "matrix_seed": 1},
        # a new matrix: tile layout, per-tile classes, first product of a host
        # vector
        {"name": "setup_spmv_poisson3d_61x67x59", "kind": "setup", "matrix": "poisson3d", "nx": 61, "ny": 67, "nz": 59, "mixed": False, "tau": 0.0},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["cg", "cg", "cg", "cg", "bicgstab", "bicgstab", "batch", "setup"])
    if kind == "batch":
        least = _log_uniform(rng, 200, 2000)
        return {"kind": "batch", "systems": rng.randint(8, 60), "nrhs": rng.choice([1, 8, 8, rng.randint(2, 7)]), "least": least,
                "most": least * rng.randint(1, 4), "matrix_seed": rng.randrange(1000)}
    mixed = rng.random() < 0.5
    case = {"kind": kind, "matrix": "poisson3d", "nx": 1, "ny": 1, "nz": 1, "mixed": mixed, "tau": 0.0}
    if kind == "bicgstab":
        m = _log_uniform(rng, 9, 96)
        case.update(matrix="convdiff3d", nx=m, ny=m, nz=m, tau=FP32_TAU if mixed else 0.0)
        return case
    if kind == "cg":
        case["matrix"] = rng.choice(["laplace2d", "poisson3d", "poisson3d", "poisson3d", "random_spd"])
    if case["matrix"] == "random_spd":
        case.update(nx=_log_uniform(rng, 3000, 200000), tau=FP32_TAU if mixed else 0.0)
    elif case["matrix"] == "laplace2d":
        side = _log_uniform(rng, 20, 260)
        case.update(nx=side, ny=max(2, side + rng.randint(-side // 4, side // 4)))
    else:
        side = _log_uniform(rng, 10, 140 if kind == "cg" else 90)
        for k in ("nx", "ny", "nz"):
            case[k] = max(2, side + rng.randint(-side // 20, side // 20))
    return case


@functools.lru_cache(maxsize=3)
def _csr(matrix, nx, ny, nz):
    if matrix == "laplace2d":
        return mf.gen_laplace2d(nx, ny)
    if matrix == "poisson3d":
        return mf.gen_poisson3d(nx, ny, nz)
    if matrix == "convdiff3d":
        return mf.gen_convdiff3d(nx, 10.0, 1.0, 0)
    return mf.gen_random_spd(nx, 2.0, 2, 2000, 0)


@functools.lru_cache(maxsize=2)
def _batch_csr(systems, least, most, matrix_seed):
    sizes = np.exp(np.random.default_rng(matrix_seed).uniform(np.log(least), np.log(most), systems))
    return [mf.gen_stencil_lognormal(2 + i % 2, int(sizes[i]), 1.5, 1000 * matrix_seed + i) for i in range(systems)]


def _rows(case):
    return case["nx"] * case["ny"] * case["nz"]


def _product(csr, x):
    rowptr, col, val = csr
    return np.add.reduceat(val * x[col], rowptr[:-1])  # every row has its diagonal


def _solution(n, seed):
    return np.random.default_rng(seed).uniform(-1.0, 1.0, n)


def _solutions(systems, nrhs, seed):
    return [np.random.default_rng([seed, i]).uniform(-1.0, 1.0, (nrhs, len(s[0]) - 1)) for i, s in enumerate(systems)]


def prepare(case, seed):
    if case["kind"] == "batch":
        systems = _batch_csr(case["systems"], case["least"], case["most"], case["matrix_seed"])
        b = [np.stack([_product(s, row) for row in x]) for s, x in zip(systems, _solutions(systems, case["nrhs"], seed))]
        return {"kind": "batch", "batch": mf.Batch(systems, case["nrhs"], tol=TOL), "b": b}
    csr = _csr(case["matrix"], case["nx"], case["ny"], case["nz"])
    n = _rows(case)
    if case["kind"] == "setup":
        return {"kind": "setup", "csr": csr, "x": _solution(n, seed), "mixed": case["mixed"]}
    A = mf.Matrix(*csr)
    A.layout(case["tau"])
    padded = A.info()["tilem"] * A.B
    b = torch.zeros(padded, dtype=torch.float64)
    b[:n] = torch.from_numpy(_product(csr, _solution(n, seed)))
    # residual replacements as the benchmark sets them for lossless and for
    # rounded tiles; FP64 replaces at convergence only
    replace = 0.0 if not case["mixed"] else 1e-4 if case["tau"] == 0.0 else 1e-2
    opts = {"tol": TOL, "maxit": 20000, "tau": case["tau"], "rr_factor": replace, "method": mf.MF_BICGSTAB if case["kind"] == "bicgstab" else mf.MF_CG,
            "precision": mf.MF_MIXED if case["mixed"] else mf.MF_FP64}
    state = {"kind": "solve", "A": A, "b": b.cuda(), "x": torch.zeros(padded, dtype=torch.float64, device="cuda"), "n": n, "opts": opts}
    torch.cuda.synchronize()  # the library works on a stream of its own
    return state


def run(state):
    if state["kind"] == "batch":
        x, _, _, _ = state["batch"].solve(state["b"])
        return {"x": [np.reshape(v, (-1, v.shape[-1])) for v in x]}
    if state["kind"] == "setup":
        A = mf.Matrix(*state["csr"])
        A.layout()
        y = A.spmv(state["x"], mixed=state["mixed"])
        codes = A.classes()
        A.close()
        return {"y": y, "codes": codes}
    report = state["A"].solve_device(state["b"].data_ptr(), state["x"].data_ptr(), **state["opts"])
    if report["status"] != 0:
        raise RuntimeError("solve: status %d" % report["status"])
    return {"x": state["x"][: state["n"]]}


def exact(case, seed):
    """The solution that b was made from: A x* is rounded once per row, which
    moves the solution of A x = b by far less than the tolerance does."""
    if case["kind"] == "batch":
        systems = _batch_csr(case["systems"], case["least"], case["most"], case["matrix_seed"])
        return {"x": _solutions(systems, case["nrhs"], seed)}
    x = _solution(_rows(case), seed)
    if case["kind"] == "setup":
        return {"y": _product(_csr(case["matrix"], case["nx"], case["ny"], case["nz"]), x), "codes": None}
    return {"x": x}


def _iterations(case):
    """Krylov iterations to the tolerance, as CG and BiCGSTAB in FP64 take
    them on these systems (fits to within some ten percent)."""
    n = _rows(case)
    if case["matrix"] == "laplace2d":
        return 3.8 * n ** 0.5
    if case["matrix"] == "poisson3d":
        return 17.5 * n ** (0.70 / 3)
    if case["matrix"] == "convdiff3d":
        return 3.65 * case["nx"]
    return 513 * (n / 30000) ** 0.234


def work(case):
    """A solve reads its matrix once per product (each nonzero's value at the
    width of its tile class, and a byte of index), and reads and writes the
    vector of that product; CG takes one product per iteration, BiCGSTAB
    two.  Set-up reads the CSR arrays and x, and writes both layouts and y."""
    if case["kind"] == "batch":
        # a 5-point (even) or 7-point (odd) stencil each, sizes log-uniform
        k = case["systems"]
        lo, hi = case["least"], case["most"]
        sizes = [lo * (hi / lo) ** ((i + 0.5) / k) for i in range(k)]
        total = flops = 0.0
        for i, n in enumerate(sizes):
            per_row, its = (5, 12 * n ** 0.5) if i % 2 == 0 else (7, 28 * n ** (1 / 3))
            total += its * n * (9 * per_row + 16 * case["nrhs"])
            flops += its * n * case["nrhs"] * (2 * per_row + 10)
        return {"bytes": total, "flops": flops}
    n = _rows(case)
    per_row = {"laplace2d": 5, "poisson3d": 7, "convdiff3d": 26.5, "random_spd": 18.2}[case["matrix"]]
    nnz = per_row * n
    if case["kind"] == "setup":
        return {"bytes": 12.0 * nnz + 4 * n + 16.0 * n + (9 + 2) * nnz, "flops": 2.0 * nnz}
    width = 8 if not case["mixed"] else 1 if case["tau"] == 0.0 else 4
    vector = 16 if not case["mixed"] else 12
    products = _iterations(case) * (2 if case["kind"] == "bicgstab" else 1)
    return {"bytes": products * (nnz * (width + 1) + vector * n), "flops": products * (2.0 * nnz + 10.0 * n)}

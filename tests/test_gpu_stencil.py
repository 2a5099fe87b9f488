"""Solves on stencil planes (matrices whose rows draw their entries from one
short list of offsets) against the same solves on the slabs, bit for bit: an
explicit index width keeps a solve on the slabs."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
TOL = 1e-10


def _banded(n, offsets, rng, drop=0.0):
    """Diagonally dominant symmetric matrix on the given positive offsets (and
    their negatives); a share of the pairs is dropped."""
    rows, cols, vals = [], [], []
    diag = np.full(n, 0.25)
    for d in offsets:
        i = np.arange(n - d)
        i = i[rng.random(len(i)) >= drop]
        v = -rng.uniform(0.5, 1.5, len(i))
        rows += [i, i + d]
        cols += [i + d, i]
        vals += [v, v]
        np.subtract.at(diag, i, v)
        np.subtract.at(diag, i + d, v)
    rows.append(np.arange(n)), cols.append(np.arange(n)), vals.append(diag)
    r, c, v = np.concatenate(rows), np.concatenate(cols), np.concatenate(vals)
    o = np.lexsort((c, r))
    rp = np.zeros(n + 1, np.int64)
    np.add.at(rp, r + 1, 1)
    return np.cumsum(rp).astype(np.int32), c[o].astype(np.int32), v[o]


def _matrix(gpu, name):
    rng = np.random.default_rng(5)
    return {
        "laplace2d_30x31": lambda: gpu.gen_laplace2d(30, 31),          # 5 offsets, one workgroup
        "laplace2d_97x83": lambda: gpu.gen_laplace2d(97, 83),          # 5 offsets, ragged last tile row
        "poisson3d_17x19x13": lambda: gpu.gen_poisson3d(17, 19, 13),   # 7 offsets
        "poisson3d_33x31x29": lambda: gpu.gen_poisson3d(33, 31, 29),
        "convdiff_14": lambda: gpu.gen_convdiff3d(14, 10.0, 1.0, 0),   # 27 offsets: quads
        "convdiff_21": lambda: gpu.gen_convdiff3d(21, 10.0, 1.0, 0),
        "lognormal_3d": lambda: gpu.gen_stencil_lognormal(3, 9000, 0.5, 3),
        "band_3": lambda: _banded(1000, (1,), rng),                    # one quad, padded
        "band_9": lambda: _banded(5003, (1, 7, 40, 41), rng),          # three quads, odd size
        "band_31": lambda: _banded(4099, tuple(range(1, 16)), rng, 0.1),
    }[name]()


CASES = [("laplace2d_30x31", 0), ("laplace2d_97x83", 0), ("laplace2d_97x83", 1), ("poisson3d_17x19x13", 0),
         ("poisson3d_33x31x29", 0), ("poisson3d_33x31x29", 3), ("convdiff_14", 0), ("convdiff_14", 2), ("convdiff_21", 0),
         ("lognormal_3d", 0), ("lognormal_3d", 2), ("band_3", 0), ("band_9", 0), ("band_9", 1), ("band_31", 0), ("band_31", 2)]


@pytest.mark.parametrize("name,grid", CASES)
@pytest.mark.parametrize("tau", [None, 0.0, 2.0 ** -24, 2.0 ** -11])
def test_gpu_planes_equal_slabs(gpu, orc, name, grid, tau):
    """Iterations and x on the planes equal those on the slabs: 5-, 7- and
    27-point stencils and bands whose tables are padded, sizes that end inside
    a tile row and a row slot, one to eight rows per thread, one workgroup and
    several, values of each class."""
    rp, ci, va = _matrix(gpu, name)
    n = len(rp) - 1
    b = orc.csr_spmv(rp, ci, va, np.random.default_rng(1).uniform(-1, 1, n))
    A, S = gpu.Matrix(rp, ci, va), gpu.Matrix(rp, ci, va)
    S.set_index_width(2)
    prec = dict(precision=gpu.MF_FP64) if tau is None else dict(precision=gpu.MF_MIXED, tau=tau, rr_factor=1e-2)
    for method in (gpu.MF_CG, gpu.MF_BICGSTAB):
        if method == gpu.MF_CG and name.startswith("convdiff"):
            continue
        o = dict(method=method, tol=TOL, grid=grid, **prec)
        print(f"case {name} grid={grid} tau={tau} method={method}", flush=True)
        x, rep = A.solve(b, **o)
        y, sep = S.solve(b, **o)
        assert rep["status"] == 0 and rep["relres_true"] <= TOL, rep
        assert (rep["iterations"], rep["replacements"], rep["grid"]) == (sep["iterations"], sep["replacements"], sep["grid"])
        assert np.array_equal(x, y)
        x2, _ = A.solve(b, **o)
        assert np.array_equal(x, x2)


def test_gpu_planes_beyond_register_x(gpu, orc):
    """17 to 36 rows per thread, where x stays in the caller's buffer (the
    vectors count as streamed): 3, 4 and 5 workgroups of 8704 to 18432 rows
    give the solution of the default grid and its iterations within one."""
    rp, ci, va = gpu.gen_poisson3d(34, 33, 32)
    n = len(rp) - 1
    b = orc.csr_spmv(rp, ci, va, np.random.default_rng(2).uniform(-1, 1, n))
    A = gpu.Matrix(rp, ci, va)
    for prec in (dict(precision=gpu.MF_FP64), dict(precision=gpu.MF_MIXED, tau=0.0, rr_factor=1e-4)):
        y, sep = A.solve(b, tol=TOL, **prec)
        for grid in (2, 3, 4):
            print(f"case poisson3d_34x33x32 grid={grid} {prec}", flush=True)
            x, rep = A.solve(b, tol=TOL, grid=grid, **prec)
            assert rep["status"] == 0 and rep["relres_true"] <= TOL and rep["streamed"] == 1
            assert abs(rep["iterations"] - sep["iterations"]) <= max(2, 0.05 * sep["iterations"])
            assert np.linalg.norm(x - y) <= 1e-8 * np.linalg.norm(y)


@pytest.mark.parametrize("name,B,grid", [
    ("poisson3d_33x31x29", 8, 0), ("poisson3d_33x31x29", 8, 54), ("laplace2d_97x83", 8, 16), ("band_9", 8, 9),
    ("poisson3d_33x31x29", 32, 0), ("laplace2d_97x83", 32, 12), ("band_9", 32, 9)])
def test_gpu_planes_replaced_residuals(gpu, orc, name, B, grid):
    """FP64 CG whose residual is replaced every two digits, on 8- and 32-row
    tiles, with several workgroups: chunks that start in the middle of a cache
    line (54 workgroups of 69 tile rows of 8 rows, 16 of 63) and odd numbers of
    tile rows.  Planes equal slabs, bit for bit."""
    rp, ci, va = _matrix(gpu, name)
    n = len(rp) - 1
    b = orc.csr_spmv(rp, ci, va, np.random.default_rng(1).uniform(-1, 1, n))
    A, S = gpu.Matrix(rp, ci, va, B=B), gpu.Matrix(rp, ci, va, B=B)
    S.set_index_width(2)
    print(f"case {name} B={B} grid={grid}", flush=True)
    o = dict(tol=TOL, grid=grid, rr_factor=1e-2)
    x, rep = A.solve(b, **o)
    y, sep = S.solve(b, **o)
    print(f"  it={rep['iterations']} repl={rep['replacements']} grid={rep['grid']}", flush=True)
    assert rep["status"] == 0 and rep["relres_true"] <= TOL and rep["replacements"] >= 4 and rep["grid"] > 1
    assert (rep["iterations"], rep["replacements"], rep["grid"]) == (sep["iterations"], sep["replacements"], sep["grid"])
    assert np.array_equal(x, y)


def test_gpu_planes_after_nonfinite_solve(gpu, orc):
    """A solve whose published FP32 entries overflowed leaves nothing behind for
    the next one on the same matrix: BiCGSTAB with neighbour waits, where
    positions that hold 0 are gathered from workgroups that are not waited for
    (the second and the fourth of four workgroups have no entry in each other's
    rows, but an offset of the table points there)."""
    n = 4096
    rng = np.random.default_rng(8)
    cols = {i: {i: -1.0 if i == n - 1 else 1.0} for i in range(n)}
    for d in (1, 2, 2048):
        for i in range(n - d):
            if d < 2048 or i < 1024:
                cols[i][i + d], cols[i + d][i] = rng.choice([-1, 1], 2) * 2.0 ** -5
    rp = np.cumsum([0] + [len(cols[i]) for i in range(n)]).astype(np.int32)
    ci = np.concatenate([sorted(cols[i]) for i in range(n)]).astype(np.int32)
    va = np.concatenate([[cols[i][c] for c in sorted(cols[i])] for i in range(n)])
    b = orc.csr_spmv(rp, ci, va, rng.uniform(-1, 1, n))
    # (b, A b) = 2^-22 (b, b), so the first step's s exceeds FP32
    bad = np.zeros(n)
    bad[1500], bad[n - 1] = 2.0 ** 120 * (1 + 2.0 ** -22), 2.0 ** 120
    o = dict(method=gpu.MF_BICGSTAB, precision=gpu.MF_MIXED, tau=0.0, rr_factor=1e-2, tol=TOL, grid=4)
    A, F = gpu.Matrix(rp, ci, va), gpu.Matrix(rp, ci, va)
    y, frep = F.solve(b, **o)
    assert frep["status"] == 0 and frep["grid"] == 4 and frep["rows_per_thread"] == 2 and 0 < frep["sync_deps"] < 4
    for turn in range(3):
        print(f"case nonfinite, then finite, turn {turn}", flush=True)
        _, rep = A.solve(bad, **o)
        assert rep["status"] in (-20, -23), rep  # breakdown, non-finite sums
        x, rep = A.solve(b, **o)
        assert rep["status"] == 0 and rep["iterations"] == frep["iterations"]
        assert np.array_equal(x, y)


@pytest.mark.parametrize("name,grid", [c for c in CASES if c[0] != "band_3"])
@pytest.mark.parametrize("tau", [None, 0.0, 2.0 ** -24, 2.0 ** -11])
def test_gpu_planes_ran(gpu, orc, name, grid, tau):
    """The solves that the comparisons above mean to run on planes do: CG on all
    of these grids, BiCGSTAB where its vectors fit on chip; none with an index
    width asked for."""
    rp, ci, va = _matrix(gpu, name)
    b = orc.csr_spmv(rp, ci, va, np.random.default_rng(1).uniform(-1, 1, len(rp) - 1))
    A, S = gpu.Matrix(rp, ci, va), gpu.Matrix(rp, ci, va)
    assert A.planes() == {"offsets": 0, "fp64": -1, "mixed": -1, "listed": 0, "ran": 0}
    prec = dict(precision=gpu.MF_FP64) if tau is None else dict(precision=gpu.MF_MIXED, tau=tau, rr_factor=1e-2)
    for method in (gpu.MF_CG, gpu.MF_BICGSTAB):
        if method == gpu.MF_CG and name.startswith("convdiff"):
            continue
        print(f"case {name} grid={grid} tau={tau} method={method}", flush=True)
        _, rep = A.solve(b, method=method, tol=TOL, grid=grid, **prec)
        p = A.planes()
        assert p["ran"] == (1 if method == gpu.MF_CG or rep["rows_per_thread"] > 0 else 0), (p, rep)
        assert p["offsets"] == len({d for i in range(len(rp) - 1) for d in ci[rp[i]:rp[i + 1]] - i})
        if p["ran"] and tau is not None:
            assert p["mixed"] in (0, 2, 3, 4) and p["listed"] == 0
        elif p["ran"]:
            assert p["fp64"] == 0 and p["mixed"] == -1
    S.solve(b, tol=TOL, index_width=2, grid=grid, **dict(prec, method=method))
    assert S.planes() == {"offsets": 0, "fp64": -1, "mixed": -1, "listed": 0, "ran": 0}


def test_gpu_planes_rows_per_thread(gpu, orc):
    """17 to 36 rows per thread: the kernels of 20, 28 and 36 rows, x in the
    caller's buffer, give the bits of the slab kernels, which stream every
    vector there."""
    rp, ci, va = gpu.gen_poisson3d(34, 33, 32)  # 35,904 rows on 4, 3 and 2 workgroups
    b = orc.csr_spmv(rp, ci, va, np.random.default_rng(2).uniform(-1, 1, len(rp) - 1))
    A, S = gpu.Matrix(rp, ci, va), gpu.Matrix(rp, ci, va)
    S.set_index_width(2)
    for prec in (dict(precision=gpu.MF_FP64), dict(precision=gpu.MF_MIXED, tau=0.0, rr_factor=1e-4)):
        for grid, rows in ((4, 20), (3, 28), (2, 36)):
            print(f"case poisson3d_34x33x32 grid={grid} {prec}", flush=True)
            x, rep = A.solve(b, tol=TOL, grid=grid, **prec)
            y, sep = S.solve(b, tol=TOL, grid=grid, **prec)
            assert A.planes()["ran"] == 1 and rep["rows_per_thread"] == rows and rep["streamed"] == 1
            assert sep["rows_per_thread"] == 0 and sep["streamed"] == 1
            assert rep["status"] == sep["status"] == 0 and rep["iterations"] == sep["iterations"]
            assert np.array_equal(x, y)


@pytest.mark.parametrize("name,tau,method,ran", [
    ("laplace2d_30x31", None, 0, 1), ("laplace2d_30x31", 2.0 ** -11, 1, 1),
    ("band_3", None, 0, 0), ("band_3", 2.0 ** -11, 1, 0),
    ("convdiff_8", None, 1, 0), ("convdiff_9", 2.0 ** -24, 1, 0), ("convdiff_9", None, 1, 1), ("convdiff_12", None, 1, 0),
    ("convdiff_12", 2.0 ** -24, 1, 1), ("convdiff_12", 2.0 ** -11, 1, 0),
    ("band_9_2000", None, 0, 0), ("band_9_2000", 2.0 ** -24, 0, 1), ("band_9_2000", 2.0 ** -11, 0, 1)])
def test_gpu_planes_one_workgroup(gpu, orc, name, tau, method, ran):
    """One workgroup runs planes of quads only where they are faster than its
    slabs (planes_serve in solver.hip), with the bits of the slabs either way."""
    if name.startswith("convdiff"):
        rp, ci, va = gpu.gen_convdiff3d(int(name.split("_")[1]), 10.0, 1.0, 0)
    else:
        rp, ci, va = _banded(2000, (1, 7, 40, 41), np.random.default_rng(5)) if name == "band_9_2000" else _matrix(gpu, name)
    b = orc.csr_spmv(rp, ci, va, np.random.default_rng(1).uniform(-1, 1, len(rp) - 1))
    A, S = gpu.Matrix(rp, ci, va), gpu.Matrix(rp, ci, va)
    S.set_index_width(2)
    prec = dict(precision=gpu.MF_FP64) if tau is None else dict(precision=gpu.MF_MIXED, tau=tau, rr_factor=1e-2)
    print(f"case {name} tau={tau} method={method}", flush=True)
    x, rep = A.solve(b, method=method, tol=TOL, **prec)
    y, sep = S.solve(b, method=method, tol=TOL, **prec)
    print(f"  it={rep['iterations']} rpt={rep['rows_per_thread']} {A.planes()}", flush=True)
    assert rep["grid"] == 1 and rep["status"] == 0 and rep["relres_true"] <= TOL
    assert A.planes()["ran"] == ran
    assert rep["iterations"] == sep["iterations"] and np.array_equal(x, y)


def test_gpu_hbm_vectors_beyond_the_slab_kernels(gpu, orc):
    """9 to 16 rows per thread on 8-row tiles: CG on planes holds the vectors,
    the slab kernels stream them, and vectors = MF_VECTORS_HBM is served by those,
    with the same bits."""
    rp, ci, va = gpu.gen_poisson3d(34, 33, 32)
    b = orc.csr_spmv(rp, ci, va, np.random.default_rng(2).uniform(-1, 1, len(rp) - 1))
    A = gpu.Matrix(rp, ci, va, B=8)
    print("case poisson3d_34x33x32 B=8 grid=5", flush=True)
    x, rep = A.solve(b, tol=TOL, grid=5)
    assert rep["status"] == 0 and rep["streamed"] == 0 and rep["rows_per_thread"] == 16 and A.planes()["ran"] == 1
    y, sep = A.solve(b, tol=TOL, grid=5, vectors=gpu.MF_VECTORS_HBM)
    assert sep["status"] == 0 and sep["streamed"] == 1 and A.planes()["ran"] == 0
    assert rep["iterations"] == sep["iterations"] and np.array_equal(x, y)
    with pytest.raises(gpu.MFError):  # 8 rows per thread: the slab kernels hold them
        A.solve(b, tol=TOL, grid=9, vectors=gpu.MF_VECTORS_HBM)


@pytest.mark.parametrize("name,grid", [
    ("laplace2d_30x31", 0), ("laplace2d_97x83", 0), ("laplace2d_97x83", 3), ("poisson3d_33x31x29", 0),
    ("poisson3d_33x31x29", 19), ("convdiff_14", 0), ("convdiff_21", 5), ("lognormal_3d", 0), ("band_9", 0), ("band_31", 0)])
@pytest.mark.parametrize("B", [8, 32])
@pytest.mark.parametrize("tau", [None, 0.0, 2.0 ** -24, 2.0 ** -11])
def test_gpu_planes_equal_slabs_tile_sizes(gpu, orc, name, grid, B, tau):
    """8- and 32-row tiles: planes and slabs sum low-precision values alike (in
    FP32 at every size), so iterations and x agree bit for bit; CG with entries
    listed beside the planes stays on the slabs."""
    rp, ci, va = _matrix(gpu, name)
    b = orc.csr_spmv(rp, ci, va, np.random.default_rng(1).uniform(-1, 1, len(rp) - 1))
    A, S = gpu.Matrix(rp, ci, va, B=B), gpu.Matrix(rp, ci, va, B=B)
    S.set_index_width(2)
    prec = dict(precision=gpu.MF_FP64) if tau is None else dict(precision=gpu.MF_MIXED, tau=tau, rr_factor=1e-2)
    for method in (gpu.MF_CG, gpu.MF_BICGSTAB):
        if method == gpu.MF_CG and name.startswith("convdiff"):
            continue
        o = dict(method=method, tol=TOL, grid=grid, **prec)
        print(f"case {name} B={B} grid={grid} tau={tau} method={method}", flush=True)
        x, rep = A.solve(b, **o)
        p = A.planes()
        y, sep = S.solve(b, **o)
        print(f"  it={rep['iterations']} slabs {sep['iterations']} rpt={rep['rows_per_thread']} {p}", flush=True)
        assert rep["status"] == 0 and rep["relres_true"] <= TOL, rep
        assert p["ran"] == (0 if p["listed"] and method == gpu.MF_CG else 1)
        assert (rep["iterations"], rep["replacements"], rep["grid"]) == (sep["iterations"], sep["replacements"], sep["grid"])
        assert np.array_equal(x, y)


def test_gpu_planes_with_listed_entries(gpu, orc):
    """A rounded layout with a few tiles of a narrower class (lognormal stencil, FP16
    tiles of 8 rows, 62 entries in E4M3): CG, which runs on its slabs, builds no
    planes for it; BiCGSTAB builds them and runs on them, and CG still does not."""
    rp, ci, va = _matrix(gpu, "lognormal_3d")
    b = orc.csr_spmv(rp, ci, va, np.random.default_rng(1).uniform(-1, 1, len(rp) - 1))
    A = gpu.Matrix(rp, ci, va, B=8)
    o = dict(tol=TOL, precision=gpu.MF_MIXED, tau=2.0 ** -11, rr_factor=1e-2)
    x, rep = A.solve(b, method=gpu.MF_CG, **o)
    assert rep["status"] == 0 and rep["fallback"] == 0
    assert A.planes() == {"offsets": 7, "fp64": -1, "mixed": -1, "listed": 62, "ran": 0}
    _, rep2 = A.solve(b, method=gpu.MF_BICGSTAB, **o)
    assert rep2["status"] == 0 and A.planes() == {"offsets": 7, "fp64": 0, "mixed": 3, "listed": 62, "ran": 1}
    y, rep3 = A.solve(b, method=gpu.MF_CG, **o)
    assert A.planes()["ran"] == 0 and rep3["iterations"] == rep["iterations"] and np.array_equal(x, y)

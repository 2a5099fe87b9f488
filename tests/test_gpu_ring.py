"""Solves whose published vector rotates through several copies against the
allocation-free solve of the same system, which has one copy and invalidates
the caches at every publish: same iterations, same bits.  The systems have an
odd number of tile rows, so that a copy of the FP32 vector is no whole number
of cache lines, and gather both ends of the vector in one workgroup."""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
TOL = 1e-10
FP32_TAU = 2.0 ** -24


def _dev(v, npad):
    d = torch.zeros(npad, dtype=torch.float64)
    d[: len(v)] = torch.from_numpy(v)
    return d.cuda()


def _periodic(m, shift, flow=0.0):
    """7-point operator on a periodic m^3 grid, planes of the third direction
    joined with a shift; flow skews the first direction."""
    n = m ** 3
    i = np.arange(n)
    x, y, z = i % m, i // m % m, i // (m * m)
    at = lambda a, b, c: a % m + m * (b % m) + m * m * (c % m)
    up = at(x + shift * (z == m - 1), y, z + 1)
    down = np.empty_like(up)
    down[up] = i
    cols = np.stack([i, at(x + 1, y, z), at(x - 1, y, z), at(x, y + 1, z), at(x, y - 1, z), up, down], axis=1)
    vals = np.tile([6.1, -1.0 + flow, -1.0 - flow, -1.0, -1.0, -1.0, -1.0], (n, 1))
    o = np.argsort(cols, axis=1)
    rp = np.arange(0, 7 * n + 1, 7, dtype=np.int32)
    return rp, np.take_along_axis(cols, o, 1).astype(np.int32).ravel(), np.take_along_axis(vals, o, 1).ravel()


def _both(gpu, orc, name, csr, B, **opts):
    rp, ci, va = csr
    n = len(rp) - 1
    b = orc.csr_spmv(rp, ci, va, np.random.default_rng(3).uniform(-1, 1, n))
    A = gpu.Matrix(rp, ci, va, B=B)
    npad = A.info()["tilem"] * B
    d_b, d_x, d_y = _dev(b, npad), _dev(b[:0], npad), _dev(b[:0], npad)
    torch.cuda.synchronize()
    print(f"case {name} n={n} B={B} {opts}", flush=True)
    rep = A.solve_device(d_b.data_ptr(), d_x.data_ptr(), tol=TOL, **opts)
    o, one = gpu.default_opts(tol=TOL, **opts), gpu.Report()
    rc = gpu.lib().mf_solve_device_noalloc(A.h, C.c_void_p(d_b.data_ptr()), C.c_void_p(d_y.data_ptr()), C.byref(o),
                                           C.byref(one))
    assert rc == 0, gpu.lib().mf_last_error().decode()
    one = one.as_dict()
    print(f"  it={rep['iterations']} one copy {one['iterations']} grid={rep['grid']} rpt={rep['rows_per_thread']}", flush=True)
    assert rep["status"] == one["status"] == 0 and rep["relres_true"] <= TOL
    assert (rep["iterations"], rep["replacements"], rep["grid"]) == (one["iterations"], one["replacements"], one["grid"])
    assert torch.equal(d_x, d_y)
    A.close()
    return rep


MIXED = dict(tau=FP32_TAU, rr_factor=1e-2)


def test_gpu_ring_random_columns(gpu, orc):
    csr = gpu.gen_random_spd(200001, 2.0, 2, 2000, 0)  # 13,313 tile rows as reordered
    rep = _both(gpu, orc, "random_spd_200001", csr, 16, precision=gpu.MF_MIXED, **MIXED)
    assert rep["reordered"] == 1 and rep["rows_per_thread"] >= 2 and rep["fallback"] == 0


@pytest.mark.parametrize("B,grid", [(8, 0), (8, 172), (16, 0), (16, 5), (32, 0)])
@pytest.mark.parametrize("kind", ["fp64", "fp32 tiles"])
def test_gpu_ring_periodic_grid(gpu, orc, B, grid, kind):
    # 61^3 = 226,981 rows: 28,373, 14,187 and 7,094 tile rows of 8, 16 and 32
    # rows, 172 workgroups of 165 of the first; 33^3: 2,247 of 16, on 5 workgroups
    # of up to 16 rows a thread
    csr = _periodic(61 if grid != 5 else 33, 17)
    prec = dict(precision=gpu.MF_FP64, rr_factor=1e-2) if kind == "fp64" else dict(precision=gpu.MF_MIXED, **MIXED)
    _both(gpu, orc, "periodic", csr, B, grid=grid, **prec)


@pytest.mark.parametrize("B", [8, 16])
def test_gpu_ring_bicgstab_grid_syncs(gpu, orc, B):
    csr = _periodic(61, 17, flow=0.25)
    _both(gpu, orc, "periodic flow", csr, B, method=gpu.MF_BICGSTAB, sync=gpu.MF_SYNC_GLOBAL, precision=gpu.MF_MIXED, **MIXED)

"""Fields and results through the solver's pinned buffers: one chunk, rows that
straddle the 1 MiB chunks, several threads, a j slab, and the paths that keep
them (cells that are not emitters keep the caller's values)."""
import ctypes as C

import numpy as np
import pytest

import dnsmc_amd
from dnsmc_amd import workloads
from dnsmc_amd._lib import check, lib

pytestmark = pytest.mark.gpu


def _fortran(S, shape):
    Q, V = np.full(shape, 7.5, np.float32, order="F"), np.full(shape, -3.25, np.float32, order="F")
    f32 = C.POINTER(C.c_float)
    check(lib().dnsmc_get_results_fortran(S.h, 0, Q.ctypes.data_as(f32), V.ctypes.data_as(f32)))
    return Q, V


@pytest.mark.parametrize("n,p_row,ystart,subset", [
    ((5, 4, 3), 1, None, 0), ((45, 61, 37), 1, None, 0), ((45, 61, 200), 1, None, 0), ((128, 64, 64), 1, None, 0),
    ((45, 62, 200), 2, 32, 0), ((45, 61, 200), 1, None, 1000),
])
def test_fields_and_results(n, p_row, ystart, subset):
    cfg = workloads.channel_config(n, rays_per_cell=2, spectral=3, Tw=300.0, kappa_grey=20.0, p_row=p_row)
    S = dnsmc_amd.Solver(cfg)
    S.load_tables()
    T = workloads.field_grey32(3, n)
    S.set_field(0, workloads.ghosted(T))
    np.testing.assert_array_equal(S.array("T", 0), T.ravel(order="F"))
    cells = None
    if subset:
        cells = np.sort(np.random.default_rng(1).choice(n[0] * n[1] * n[2], subset, replace=False)).astype(np.int32)
        S.set_emitters(cells)
    if ystart is not None:
        check(lib().dnsmc_set_emitters_slab(S.h, ystart))
    S.run()
    S.wait()
    nj = n[1] // p_row
    ne = subset or n[0] * nj * n[2]
    res = {k: np.full(ne, np.nan) for k in ("Q", "E", "A", "sdev")}
    f64 = C.POINTER(C.c_double)
    check(lib().dnsmc_get_results(S.h, 0, *[res[k].ctypes.data_as(f64) for k in ("Q", "E", "A", "sdev")]))
    assert all(np.isfinite(v).all() for v in res.values())
    np.testing.assert_allclose(res["Q"], res["E"] - res["A"], rtol=0, atol=1e-9 * np.max(res["E"]))
    Q, V = _fortran(S, (n[0] + 2, nj + 2, n[2] + 2))
    for got, want, ghost in ((Q, res["Q"], 7.5), (V, res["sdev"], -3.25)):
        ref = np.full(got.shape, ghost, np.float32, order="F")
        inner = np.full(n[0] * nj * n[2], ghost, np.float32)
        inner[cells if subset else slice(None)] = want.astype(np.float32)
        ref[1:-1, 1:-1, 1:-1] = inner.reshape((n[0], nj, n[2]), order="F")
        np.testing.assert_array_equal(got, ref)

"""Results at the sizes where their copies change: plain below 4 MiB in one call,
several threads from there on (the FP32 rows of the Fortran layout: one thread
below).  The same arrays fetched one by one pass the other path.  Bits equal."""
import ctypes as C

import numpy as np
import pytest

import dnsmc_amd
from dnsmc_amd import workloads
from dnsmc_amd._lib import check, lib

pytestmark = pytest.mark.gpu
KEYS = ("Q", "E", "A", "sdev")


# four FP64 arrays: 32 bytes per cell
@pytest.mark.parametrize("n,total", [((2, 2, 2), 256), ((64, 32, 32), 2 << 20), ((63, 65, 32), 4193280), ((64, 64, 32), 4 << 20),
                                     ((65, 64, 32), 4259840), ((128, 64, 64), 16 << 20), ((129, 64, 64), 16908288)])
def test_results_at_the_edges(n, total):
    cfg = workloads.channel_config(n, rays_per_cell=2, spectral=3, Tw=300.0, kappa_grey=20.0)
    S = dnsmc_amd.Solver(cfg)
    S.load_tables()
    T = workloads.field_grey32(3, n)
    S.set_field(0, workloads.ghosted(T))
    np.testing.assert_array_equal(S.array("T", 0), T.ravel(order="F"))
    S.run()
    ne = n[0] * n[1] * n[2]
    assert 32 * ne == total
    f64 = C.POINTER(C.c_double)

    def fetch(keys):
        out = {k: np.full(ne, np.nan) for k in keys}
        check(lib().dnsmc_get_results(S.h, 0, *[out[k].ctypes.data_as(f64) if k in keys else None for k in KEYS]))
        return out

    every = fetch(KEYS)
    for k in KEYS:
        assert np.isfinite(every[k]).all()
        np.testing.assert_array_equal(fetch((k,))[k], every[k])
    three = fetch(KEYS[1:])
    for k in KEYS[1:]:
        np.testing.assert_array_equal(three[k], every[k])
    Q = S.results_fortran(0)[0]
    np.testing.assert_array_equal(np.asarray(Q)[1:-1, 1:-1, 1:-1], every["Q"].reshape(n, order="F").astype(np.float32))
    S.close()

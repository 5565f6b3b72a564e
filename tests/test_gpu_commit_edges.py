"""Committing a field where the spline and range passes can go wrong: lines of
2 to 130 values (groups of 16, their remainders), line counts off 64, coarse
counts off 16, bricks that the domain fills in part, one to four coarse levels.

Coarse fields equal the oracle's FP64 spline to 2e-7 (the FP32 rounding of the
result); the range is the fields' own: Tmax, a negative value in any corner, and
where the table slice fits LDS its nodes, which follow from the smallest and
largest value with the kernel's own FP32 coordinate."""
import numpy as np
import pytest

import dnsmc_amd
from dnsmc_amd import workloads
from dnsmc_amd._lib import DnsmcError

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,levels", [((2, 2, 4), 2), ((4, 6, 2), 2), ((16, 18, 34), 2), ((36, 20, 68), 3), ((130, 6, 10), 2),
                                      ((32, 48, 16), 5), ((5, 7, 3), 1)])
def test_levels_and_range(oracle, ck_table_dir, n, levels):
    cfg = workloads.channel_config(n, rays_per_cell=2, spectral=0, Tw=573.0, grid_num=levels, table_dir=ck_table_dir[0])
    S = dnsmc_amd.Solver(cfg)
    S.load_tables()
    T = (700.0 + 40.0 * np.random.default_rng(8).standard_normal(n).clip(-3, 3)).astype(np.float32)
    T[-1, -1, -1], T[0, -1, 0] = 930.0, 410.0
    S.set_field(0, workloads.ghosted(T))
    S.run()
    st = S.stats()
    fine = [S.array("centres%d" % a, 0) for a in range(3)]
    T0 = S.array("T", 0)
    np.testing.assert_array_equal(T0, T.ravel(order="F"))
    every = [T0]
    for l in range(1, levels):
        fc = [S.array("centres%d" % a, l) for a in range(3)]
        nc = [len(c) - 2 for c in fc]
        ref = oracle.interp3d(list(n), fine[0], fine[1], fine[2], T0, nc, fc[0], fc[1], fc[2])
        every.append(S.array("T", l))
        np.testing.assert_allclose(every[-1], ref, rtol=2e-7, atol=0)
    assert st["Tmax"] == np.float32(930.0)
    sc = S.array("scalars")
    nT, inv_dT, mT0 = int(sc[5]), np.float64(sc[6]), np.float64(sc[7])

    def node(t):
        pos = np.float32(np.float64(t) * inv_dT + mT0)        # one rounding, as fmaf
        return min(int(min(max(pos, np.float32(0)), np.float32(nT - 1))), nT - 2)

    lo, hi = min(v.min() for v in every), max(v.max() for v in every)
    if st["table_mode"] == 2:   # the slice fits LDS beside this grid's faces; else the whole table counts
        assert (st["table_lo"], st["table_nw"]) == (node(lo), node(hi) + 2 - node(lo))
    else:
        assert (st["table_lo"], st["table_nw"]) == (0, nT)
    # the smallest value of every corner is seen
    for c in ((0, 0, 0), (-1, 0, 0), (0, -1, -1), (-1, -1, -1)):
        bad = T.copy()
        bad[c] = -1.0
        with pytest.raises(DnsmcError):
            S.set_field(0, workloads.ghosted(bad))

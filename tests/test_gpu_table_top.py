"""Temperatures at the top of the spectral table: the fine field stays below the
last node, the spline of a coarse level overshoots it.  The lookups clamp there
and the solve keeps its tables in LDS.

Tolerances: steps, end type and visited cells exact; D and G as the other parity
tests.  Between the table placements only the clamped cells differ, by the
rounding of k0 + 1 (k1 - k0) against k1 (6e-8 of kappa and of Ib, so about as
much of a ray's E and A; 1e-6 allowed).
"""
import numpy as np
import pytest

import dnsmc_amd
from dnsmc_amd import workloads
from helpers import oracle_problem_dict

pytestmark = pytest.mark.gpu
N, R, MAXS = (8, 12, 8), 16, (3, 100000, 100000, 100000, 100000, 100000)


def _field():
    """1850 K with pairs of cells (a coarse cell each) at 1996 K: the spline between them reaches 2014 K."""
    T = np.full(N, 1850.0, np.float32)
    T[2:4] = 1996.0
    T[6:8] = 1996.0
    return T


@pytest.mark.parametrize("top", [1996.0, 1950.0])
def test_coarse_level_above_the_table(oracle, ck_table_dir, monkeypatch, top):
    T = np.where(_field() > 1900.0, np.float32(top), _field())
    cfg = workloads.channel_config(N, rays_per_cell=R, spectral=0, Tw=573.0, grid_num=2, maxs=MAXS,
                                   table_dir=ck_table_dir[0])
    nT, last = 69, 2000.0
    res = {}
    for tables in ("", "global"):
        monkeypatch.setenv("DNSMC_TABLES", tables)
        S = dnsmc_amd.Solver(cfg)
        S.load_tables()
        S.set_field(0, workloads.ghosted(T))
        assert np.max(S.array("T", 0)) < last and (np.max(S.array("T", 1)) > last) == (top == 1996.0)
        S.run()
        res[tables], st = S.results(0), S.stats()
        assert st["table_mode"] == (0 if tables else 2)
        if not tables:
            assert st["table_lo"] + st["table_nw"] <= nT
            S.set_record(True)
            S.run()
            assert S.stats()["table_mode"] == 2 and S.stats()["n_steps"] == st["n_steps"]
            rec = S.records(S.nemit * R)
            d = oracle_problem_dict(S, cfg)
            P = oracle.problem(d)
            ib = float(np.max(d["Ib"]))
            for cell in range(0, S.nemit, 7):
                ref = oracle.gen_philox(P, cfg.seed, 0, cell, 0, R)
                i, j, k = cell % N[0] + 1, (cell // N[0]) % N[1] + 1, cell // (N[0] * N[1]) + 1
                for r in range(R):
                    w0, w1 = int(ref["w0"][r]), int(ref["w1"][r])
                    u = [(float(w & 0xFFFFFF) + d["u_off"]) * 2.0 ** -24 for w in (w0, w1)]
                    o = oracle.trace_ray(P, i, j, k, u[0], u[1], (w0 >> 24) | (((w1 >> 24) & 3) << 8), w1 >> 26)
                    q = cell * R + r
                    assert (rec["steps"][q], rec["end"][q], rec["hash"][q]) == (o.steps, o.end_type, o.hash), (cell, r)
                    assert abs(rec["D"][q] - o.D) <= 2e-5 * max(abs(o.D), 1e-30), (cell, r)
                    assert abs(rec["G"][q] - o.G) <= 2e-5 * abs(o.G) + 5e-6 * ib, (cell, r)
        S.close()
    for key in ("E", "A"):
        np.testing.assert_allclose(res[""][key], res["global"][key], rtol=1e-6, atol=0)

"""The FP64 traversal's hand-out and drain (kDrain = 16 crossings per batch):
launches of less than a claim, domains of 1 to 5 cells (a periodic wrap or a
wall in every batch), step caps around multiples of the batch, three levels.

Step totals equal the oracle's.  E and A follow the oracle's
FP64 estimator to 1e-12: only the last bits of sin, cos and exp differ, 1e-16
each, over chains of at most 1e5 additions of positive terms whose rounding is
the same on both sides."""
import numpy as np
import pytest

import dnsmc_amd
from dnsmc_amd import workloads
from helpers import oracle_problem_dict

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,levels,maxs,kappa,R", [
    ((1, 2, 1), 1, (16,), 0.02, 2),
    ((1, 2, 1), 1, (16,), 0.02, 3),
    ((3, 2, 5), 1, (17,), 0.02, 5),
    ((5, 4, 3), 1, (3000,), 0.3, 40),
    ((4, 3, 2), 1, (3000,), 1e-4, 17),
    ((8, 8, 4), 3, (5, 3, 3000), 0.01, 7),
    ((8, 4, 8), 3, (1, 15, 31), 0.01, 7),
    ((12, 16, 9), 1, (33,), 0.05, 700),
])
@pytest.mark.parametrize("spectral", [3, 0])
def test_f64_rays_match_oracle(oracle, ck_table_dir, n, levels, maxs, kappa, R, spectral):
    maxs = tuple(maxs) + (3000,) * (6 - len(maxs))
    cfg = workloads.channel_config(n, rays_per_cell=R, spectral=spectral, Tw=300.0 if spectral == 3 else 573.0,
                                   grid_num=levels, maxs=maxs, kappa_grey=kappa, table_dir=ck_table_dir[0],
                                   precision=1, tally=1)
    S = dnsmc_amd.Solver(cfg)
    S.load_tables()
    T = (700.0 + 40.0 * np.random.default_rng(4).standard_normal(n).clip(-3, 3)).astype(np.float32)
    S.set_field(0, workloads.ghosted(T))
    S.set_record(True)
    S.run()
    res, st = S.results(0), S.stats()
    rec = S.records(S.nemit * R)
    P = oracle.problem(oracle_problem_dict(S, cfg))
    E, A, Q2, ns = oracle.mc_philox(P, cfg.seed, 0, R, f64=True)
    assert st["n_steps"] == ns and int(np.sum(rec["steps"])) == ns
    np.testing.assert_allclose(res["E"], E, rtol=1e-12, atol=0)
    np.testing.assert_allclose(res["A"], A, rtol=1e-12, atol=0)
    S.set_record(False)
    S.run()
    res2, st2 = S.results(0), S.stats()
    assert st2["n_steps"] == ns
    np.testing.assert_array_equal(res2["E"], res["E"])
    np.testing.assert_array_equal(res2["A"], res["A"])

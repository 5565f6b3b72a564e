"""The FP64 traversal's hand-out of rays: eight shares, the first chunk of a wave
by its place, the rest claimed (kappa 0.02: up to thousands of crossings), or a
thread per ray (kappa 2: some fifty at most).  Launches of fewer rays than a share's rounding,
of one block and of shares that other XCDs' waves have to empty, to several
claims per wave, against the oracle's FP64 estimator (step totals equal, E and A
to 1e-12: the last bits of sin, cos and exp in sums of positive terms)."""
import numpy as np
import pytest

import dnsmc_amd
from dnsmc_amd import workloads
from helpers import oracle_problem_dict

pytestmark = pytest.mark.gpu
N = (8, 12, 8)


@pytest.mark.parametrize("cells,R", [(1, 2), (1, 64), (1, 65), (3, 85), (1, 511), (2, 256), (5, 409), (9, 1000), (130, 257),
                                     (768, 300)])
@pytest.mark.parametrize("kappa", [2.0, 0.02])
@pytest.mark.parametrize("levels", [1, 3])
def test_every_ray_once(oracle, cells, R, levels, kappa):
    cfg = workloads.channel_config(N, rays_per_cell=R, spectral=3, Tw=300.0, kappa_grey=kappa, grid_num=levels,
                                   maxs=(5, 5, 3000, 3000, 3000, 3000) if levels > 1 else (3000,) * 6, precision=1, tally=1)
    S = dnsmc_amd.Solver(cfg)
    S.load_tables()
    S.set_field(0, workloads.ghosted(workloads.field_grey32(5, N)))
    some = np.sort(np.random.default_rng(2).choice(768, cells, replace=False)).astype(np.int32)
    S.set_emitters(some)
    S.run()
    res, st = S.results(0), S.stats()
    P = oracle.problem(oracle_problem_dict(S, cfg))
    E, A, Q2, ns = oracle.mc_philox(P, cfg.seed, 0, R, cells=some, f64=True)
    assert st["n_steps"] == ns
    np.testing.assert_allclose(res["E"], E, rtol=1e-12, atol=0)
    np.testing.assert_allclose(res["A"], A, rtol=1e-12, atol=0)
    S.close()

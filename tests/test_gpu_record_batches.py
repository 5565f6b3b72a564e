"""Recorded runs of several batches or snapshots: only the first batch of
snapshot 0 is recorded, the launches after it trace from the ray queue.  E, A
and the step count against the same run without records.

Sizes: grids whose faces and offsets are smaller than a block's tally ring
(1 KiB for four waves) and one whose tables fill LDS beside it; the rays are the
same, the FP64 sums in another order (1e-12).
"""
import numpy as np
import pytest

import dnsmc_amd
from dnsmc_amd import workloads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,spectral,R,batch,nsnap,tally", [
    ((24, 1, 5), 3, 257, 5000, 1, 0),
    ((4, 3, 2), 3, 100, 1024, 1, 0),
    ((3, 2, 5), 3, 40, 1 << 30, 2, 0),
    ((8, 8, 4), 0, 64, 1024, 2, 0),
    ((12, 16, 9), 0, 33, 1 << 30, 3, 0),
    ((5, 6, 7), 3, 50, 1024, 2, 1),
])
def test_recorded_runs_of_several_launches(ck_table_dir, monkeypatch, n, spectral, R, batch, nsnap, tally):
    cfg = workloads.channel_config(n, rays_per_cell=R, spectral=spectral, Tw=300.0 if spectral == 3 else 573.0,
                                   nsnap=nsnap, kappa_grey=0.05, table_dir=ck_table_dir[0])
    cfg.batch_rays = batch
    cfg.tally = tally
    for tables in ("", "global"):
        monkeypatch.setenv("DNSMC_TABLES", tables)
        S = dnsmc_amd.Solver(cfg)
        S.load_tables()
        rng = np.random.default_rng(2)
        for s in range(nsnap):
            T = (700.0 + 40.0 * rng.standard_normal(n).clip(-3, 3)).astype(np.float32)
            S.set_field(s, workloads.ghosted(T))
        S.run()
        want, steps = [S.results(s) for s in range(nsnap)], S.stats()["n_steps"]
        S.set_record(True)
        S.run()
        got = [S.results(s) for s in range(nsnap)]
        assert S.stats()["n_steps"] == steps
        for w, g in zip(want, got):
            for key in ("E", "A"):
                np.testing.assert_allclose(g[key], w[key], rtol=1e-12, atol=0)
        S.close()

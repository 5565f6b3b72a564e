"""Reference sampling at the edges of the generators' runs, staging pieces and
chunks: every descriptor bit for bit against the oracle's sequential replay."""
import numpy as np
import pytest

import dnsmc_amd
from dnsmc_amd import workloads
from helpers import oracle_problem_dict, read_reference_tables, ref_subsequence

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("photmax", [1, 3, 4, 63, 65, 513, 1025, 2048, 2049, 4097, 9000])
@pytest.mark.parametrize("sobol", [1, 0])
@pytest.mark.parametrize("srt", [0, 1])
def test_compat_descriptors(oracle, ck_table_dir, srt, sobol, photmax):
    tdir, _ = ck_table_dir
    n, nvar = (16, 3, 2), 3
    cfg = workloads.channel_config(n, spectral=0, Tw=573.0, table_dir=tdir, mode=1, srt=srt, sobol=sobol,
                                   photmax=photmax, nvar=nvar, num_streams=16)
    S = dnsmc_amd.Solver(cfg)
    S.load_tables()
    S.set_field(0, workloads.ghosted(workloads.field_profile_noise(7, n)))
    S.run()
    S.wait()
    P = oracle.problem(oracle_problem_dict(S, cfg))
    order = oracle.sort_idx(read_reference_tables(tdir, gas=True)["kavg"])
    rays = S.rays(S.nemit * nvar * photmax)
    for cell in [0, 15, 50, 95]:
        i, j, k = cell % n[0], (cell // n[0]) % n[1], cell // (n[0] * n[1])
        for v in range(nvar):
            sub = ref_subsequence(i, j, k, v, n)
            if srt:
                ref = oracle.gen_compat_sorted(P, cfg.seed, sub, sobol, v * photmax, cell, photmax, order)
            else:
                ref = oracle.gen_compat(P, cfg.seed, sub, sobol, v * photmax, cell, photmax)
            q0 = (cell * nvar + v) * photmax
            got = rays[q0:q0 + photmax]
            np.testing.assert_array_equal(got["w0"], ref["w0"])
            np.testing.assert_array_equal(got["w1"], ref["w1"])
            np.testing.assert_allclose(got["w"], ref["w"], rtol=2e-7)


@pytest.mark.parametrize("photmax", [255, 256, 257, 700, 5000])
@pytest.mark.parametrize("levels", [1, 2])
def test_shared_slot_tallies(ck_table_dir, levels, photmax):
    """The tallies of launches with 256 rays per slot and more (16 lanes' sums at
    a time) and less, against the ordered FP64 sums of the same rays: only the
    order of FP64 additions differs."""
    res = {}
    for tally in (0, 1):
        cfg = workloads.channel_config((16, 4, 4), spectral=0, Tw=573.0, table_dir=ck_table_dir[0], mode=1, srt=0, sobol=1,
                                       photmax=photmax, nvar=3, num_streams=16, grid_num=levels, tally=tally)
        S = dnsmc_amd.Solver(cfg)
        S.load_tables()
        S.set_field(0, workloads.ghosted(workloads.field_profile_noise(7, (16, 4, 4))))
        S.run()
        res[tally] = (S.results(0), S.stats()["n_steps"])
    assert res[0][1] == res[1][1]
    for k in ("E", "A"):
        np.testing.assert_allclose(res[0][0][k], res[1][0][k], rtol=1e-11, atol=0)

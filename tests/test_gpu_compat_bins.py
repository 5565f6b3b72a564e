"""Reference sampling with tables near the largest that its generator takes: the
g CDFs in LDS (512 bands, up to 99 % of it) and from memory (628 bands: the staged
descriptors leave them no room).  Descriptors bit for bit against the
oracle's sequential replay.  One band more than fits is refused."""
import numpy as np
import pytest

import dnsmc_amd
from dnsmc_amd import workloads
from dnsmc_amd._lib import DnsmcError
from helpers import oracle_problem_dict, ref_subsequence

pytestmark = pytest.mark.gpu
N, NVAR = (16, 3, 2), 2


def _solver(nB, nQ, photmax, sobol):
    t = workloads.table_arrays(workloads.synth_ck_table(7, nB=nB, nQ=nQ, dT=50.0))
    cfg = workloads.channel_config(N, spectral=0, Tw=573.0, mode=1, srt=0, sobol=sobol, photmax=photmax, nvar=NVAR,
                                   num_streams=16)
    S = dnsmc_amd.Solver(cfg)
    S.set_tables(t)
    S.set_field(0, workloads.ghosted(workloads.field_profile_noise(7, N)))
    return S, cfg


# words of LDS: 232 + 18 (34 beyond 2048 bundles) x threads + 2 nB, + nB nQ for the g CDFs, of 40960
@pytest.mark.parametrize("nB,nQ,photmax", [(512, 64, 100), (512, 64, 2048), (512, 64, 2049), (628, 64, 700), (628, 64, 5000)])
@pytest.mark.parametrize("sobol", [1, 0])
def test_large_tables(oracle, nB, nQ, photmax, sobol):
    S, cfg = _solver(nB, nQ, photmax, sobol)
    S.run()
    S.wait()
    P = oracle.problem(oracle_problem_dict(S, cfg))
    rays = S.rays(S.nemit * NVAR * photmax)
    for cell in (0, 15, 50, 95):
        i, j, k = cell % N[0], (cell // N[0]) % N[1], cell // (N[0] * N[1])
        for v in range(NVAR):
            ref = oracle.gen_compat(P, cfg.seed, ref_subsequence(i, j, k, v, N), sobol, v * photmax, cell, photmax)
            got = rays[(cell * NVAR + v) * photmax:][:photmax]
            np.testing.assert_array_equal(got["w0"], ref["w0"])
            np.testing.assert_array_equal(got["w1"], ref["w1"])
            np.testing.assert_allclose(got["w"], ref["w"], rtol=2e-7)
    S.close()


def test_one_band_too_many():
    S, _ = _solver(630, 64, 64, 1)           # 630 x 65 + 64 words
    with pytest.raises(DnsmcError):
        S.run()
    S.close()

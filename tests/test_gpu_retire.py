"""Waves that stop claiming rays while they hold a long one: forced at any time
beyond 2 crossings (DNSMC_RETIRE=2) in launches of several claims per wave,
against launches in which no wave may (0).  Every ray is traced once either way:
step totals equal, tallies equal up to the order of their FP64 additions (1e-12;
the ordered sums bit for bit)."""
import numpy as np
import pytest

import dnsmc_amd
from dnsmc_amd import workloads

pytestmark = pytest.mark.gpu
N, R = (48, 64, 48), 32          # 4.7 million rays, super-chunks of 64: some 18 claims per resident wave


@pytest.mark.parametrize("spectral,levels,kw,env", [
    (0, 1, {}, {"DNSMC_LONG_FIRST": "0"}),                      # drawn in the traversal
    (0, 1, {}, {}),                                             # ... with the list of long rays
    (0, 2, dict(nsnap=2), {}),
    (3, 1, dict(kappa_grey=0.3), {}),
    (0, 1, {}, {"DNSMC_FUSED": "0"}),                           # from descriptors
    (0, 2, dict(tally=1), {}),                                  # the ordered sums' hand-out
])
def test_retiring_waves_lose_no_ray(ck_table_dir, monkeypatch, spectral, levels, kw, env):
    monkeypatch.setenv("DNSMC_SUPER", "64")
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    cfg = workloads.channel_config(N, rays_per_cell=R, spectral=spectral, Tw=573.0 if spectral == 0 else 300.0,
                                   table_dir=ck_table_dir[0], grid_num=levels, maxs=(6,) + (100000,) * 5 if levels > 1
                                   else (100000,) * 6, **kw)
    out = {}
    for retire in ("0", "2"):
        monkeypatch.setenv("DNSMC_RETIRE", retire)
        S = dnsmc_amd.Solver(cfg)
        S.load_tables()
        for s in range(cfg.nsnap):
            T = workloads.field_fourier(30 + s, N) if spectral == 0 else workloads.field_grey32(30 + s, N)
            S.set_field(s, workloads.ghosted(T))
        S.run()
        st = S.stats()
        asked = S.array("retired")
        assert (asked[0] > 0) == (retire == "2"), asked
        if not env and not kw and spectral == 0:
            assert st["n_listed"] > 0
        out[retire] = (st, [S.results(s) for s in range(cfg.nsnap)])
        S.close()
    (s0, r0), (s1, r1) = out["0"], out["2"]
    assert s0["n_steps"] == s1["n_steps"]
    for a, b in zip(r0, r1):
        for key in ("E", "A"):
            if kw.get("tally") == 1:
                np.testing.assert_array_equal(a[key], b[key])
            else:
                np.testing.assert_allclose(a[key], b[key], rtol=1e-12, atol=0)

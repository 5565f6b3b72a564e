"""The list of long rays where the solver would not form it by itself: launches
in which every ray starts at once, and grey gas of few crossings, with
DNSMC_LONG_FIRST=1; and the overflow of a list that, with room, is formed.
Every ray is traced once: step totals equal, tallies up to the order of their
FP64 additions."""
import numpy as np
import pytest

import dnsmc_amd
from dnsmc_amd import workloads

pytestmark = pytest.mark.gpu


def _solve(cfg, spectral, monkeypatch, env):
    for k in ("DNSMC_LONG_FIRST", "DNSMC_LONG_CAP"):
        monkeypatch.delenv(k, raising=False)
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    n = tuple(cfg.n)
    S = dnsmc_amd.Solver(cfg)
    S.load_tables()
    for s in range(cfg.nsnap):
        T = workloads.field_fourier(80 + s, n) if spectral == 0 else workloads.field_grey32(80 + s, n)
        S.set_field(s, workloads.ghosted(T))
    S.run()
    out = S.stats(), [S.results(s) for s in range(cfg.nsnap)]
    S.close()
    return out


def _same(a, b):
    assert a[0]["n_steps"] == b[0]["n_steps"]
    for x, y in zip(a[1], b[1]):
        np.testing.assert_allclose(x["E"], y["E"], rtol=1e-12, atol=0)
        np.testing.assert_allclose(x["A"], y["A"], rtol=1e-12, atol=0)


@pytest.mark.parametrize("spectral,levels,R", [(0, 1, 8), (0, 2, 30), (3, 1, 8), (3, 1, 100)])
def test_list_on_request(ck_table_dir, monkeypatch, spectral, levels, R):
    monkeypatch.setenv("DNSMC_SUPER", "64")
    cfg = workloads.channel_config((16, 24, 16), rays_per_cell=R, spectral=spectral, Tw=573.0 if spectral == 0 else 300.0,
                                   table_dir=ck_table_dir[0], grid_num=levels, maxs=(6,) + (100000,) * 5 if levels > 1
                                   else (100000,) * 6)
    own = _solve(cfg, spectral, monkeypatch, {})
    off = _solve(cfg, spectral, monkeypatch, {"DNSMC_LONG_FIRST": "0"})
    on = _solve(cfg, spectral, monkeypatch, {"DNSMC_LONG_FIRST": "1"})
    assert own[0]["n_listed"] == off[0]["n_listed"] == 0
    # 2 % of the rays of the final quarter of each XCD's share
    assert 0.01 * 0.25 * 6144 * R < on[0]["n_listed"] < 0.03 * 0.3 * 6144 * R
    _same(on, off)
    _same(own, off)


def test_overflow_of_a_list_that_fits_otherwise(ck_table_dir, monkeypatch):
    monkeypatch.setenv("DNSMC_SUPER", "512")
    cfg = workloads.channel_config((16, 24, 16), rays_per_cell=48, spectral=0, Tw=573.0, table_dir=ck_table_dir[0], nsnap=2)
    room = _solve(cfg, 0, monkeypatch, {"DNSMC_LONG_FIRST": "1"})
    capped = _solve(cfg, 0, monkeypatch, {"DNSMC_LONG_FIRST": "1", "DNSMC_LONG_CAP": "8"})
    assert room[0]["n_listed"] > 0 and capped[0]["n_listed"] == 0
    _same(room, capped)

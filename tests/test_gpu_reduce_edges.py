"""The ordered per-slot sums (tally 1: FP64, 2: Kahan-compensated FP32, 3: FP32)
at the edges of a block's slots (16, 64) and rays per tile (64, 16): equal, bit
for bit, to the same additions of the recorded rays' contributions in numpy."""
import numpy as np
import pytest

import dnsmc_amd
from dnsmc_amd import workloads

pytestmark = pytest.mark.gpu


def _sums(e, a, tally):
    """e, a: [slot][ray] float32 contributions."""
    n, R = e.shape
    if tally == 1:
        s = [np.zeros(n), np.zeros(n)]
        for r in range(R):
            s[0] = s[0] + e[:, r].astype(np.float64)
            s[1] = s[1] + a[:, r].astype(np.float64)
        return s
    out = []
    for x in (e, a):
        s, c = np.zeros(n, np.float32), np.zeros(n, np.float32)
        for r in range(R):
            if tally == 2:
                y = x[:, r] - c
                t = s + y
                c = (t - s) - y
                s = t
            else:
                s = s + x[:, r]
        out.append(s.astype(np.float64))
    return out


@pytest.mark.parametrize("tally", [1, 2, 3])
@pytest.mark.parametrize("n,R", [((1, 2, 1), 2), ((3, 5, 1), 63), ((4, 2, 2), 64), ((4, 2, 2), 65), ((17, 1, 1), 1025),
                                 ((32, 32, 16), 15), ((33, 32, 16), 17)])
def test_ordered_sums(n, R, tally):
    cfg = workloads.channel_config(n, rays_per_cell=R, spectral=3, Tw=300.0, kappa_grey=2.0, tally=tally)
    S = dnsmc_amd.Solver(cfg)
    S.load_tables()
    S.set_field(0, workloads.ghosted(workloads.field_grey32(3, n)))
    S.set_record(True)
    S.run()
    N = S.nemit
    rays, rec = S.rays(N * R), S.records(N * R)
    e = (rays["w"] * rec["D"]).reshape(N, R)
    a = (rays["winv"] * rec["G"]).reshape(N, R)
    S.set_record(False)
    S.run()
    res = S.results(0)
    E, A = _sums(e, a, tally)
    np.testing.assert_array_equal(res["E"], E)
    np.testing.assert_array_equal(res["A"], A)

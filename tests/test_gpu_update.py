"""The update of zones whose rows fill no strip, one strip or several, with the
inflation, a clamp per element and FP64 and FP32 members, against the oracle.
Needs an MI355X."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.kfcheck import rel_err
from tests.test_gpu_coverage import TOL64, TOL_MIXED, ensemble_errors

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [[1, 2, 15, 16, 17, 3], [15, 16, 17, 33, 64, 65, 20, 40],
                                  [64, 65, 129, 130, 200, 16]])
@pytest.mark.parametrize("N", [2, 7, 16, 17, 31, 32, 33, 50, 64, 65, 100, 128, 150, 256])
def test_update_vs_oracle(N, rows):
    from oak_amd import assimilation as A
    g = np.random.default_rng(N + len(rows))
    zone_ptr = np.cumsum(np.r_[0, rows]).astype(np.int64)
    n, nz, m = int(zone_ptr[-1]), len(rows), 12
    zpos = np.zeros((nz, 4))
    zpos[:, 0] = np.arange(nz)
    L, cut = np.full(nz, 2.0), np.full(nz, 2.5)
    ox, oy = np.r_[g.uniform(-0.5, nz - 3.0, m)], np.zeros(m)  # none in reach of the last zone
    ox = np.minimum(ox, nz - 3.6)
    Hj = g.integers(0, n, m).astype(np.int32)
    Hi, Hs, sh = np.arange(m, dtype=np.int32), np.ones(m), np.zeros(m)
    E = np.asfortranarray(5.0 + g.standard_normal((n, N)))
    yo, r2 = 5.0 + g.standard_normal(m), np.full(m, 0.3)
    mc = np.where(np.arange(n) % 3 == 0, 0.05, 10.0)
    geo = A.Geometry(zone_ptr, zpos, L, cut, ox, oy, metric=0, loctype=1)
    gd = dict(zone_ptr=zone_ptr, zpos=zpos, L=L, cutoff=cut, metric=0, loctype=1, ox=ox, oy=oy)
    Eo, xo, cnt = O.ensemble_analysis(gd, (Hi, Hj, Hs), sh, yo, r2, E, inflation=1.1,
                                      max_correction=mc)
    assert cnt[-1] == 0 and cnt[0] > 0
    xf = E.mean(axis=1)
    H = A.coo_to_csr(m, Hi, Hj, Hs)
    Ea = A.ensemble_analysis(geo, H, sh, yo, r2, E, inflation=1.1, max_correction=mc)
    assert rel_err(Ea - xf[:, None], Eo - xf[:, None]) < TOL64
    Ea = A.ensemble_analysis(geo, H, sh.astype(np.float32), yo, r2, E.astype(np.float32),
                             inflation=1.1, max_correction=mc)
    e = ensemble_errors(Ea, Eo, E)
    assert e["mean_err"] < TOL_MIXED and e["spread_err"] < TOL_MIXED, e

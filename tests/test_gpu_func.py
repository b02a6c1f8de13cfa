"""M^-1/2, a and v from the tridiagonal form at the ensemble sizes where the
kernels' tiles, halves and reflector blocks end, for zones with no, few and many
observations and for small and large condition numbers, against the oracle.
Needs an MI355X."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.kfcheck import rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sigma", [0.5, 2e-3])
@pytest.mark.parametrize("N", [1, 2, 3, 15, 16, 17, 18, 31, 32, 33, 47, 64, 65, 97, 127, 128,
                               129, 144, 145, 192, 193, 194, 200, 255, 256])
def test_functions_vs_oracle(N, sigma):
    from oak_amd.rrsqrt import loc_analysis_csr
    g = np.random.default_rng(N)
    p = np.array([0, 1, 2, 3, max(N - 1, 1), N, N + 1, 3 * N, 150, 511, 512, 600])
    m = int(p.max())
    nz = len(p)
    zone_ptr = np.cumsum(np.r_[0, 1 + np.arange(nz) % 3])
    n = int(zone_ptr[-1])
    sel_ptr = np.r_[0, np.cumsum(p)]
    sel_idx = np.concatenate([np.sort(g.permutation(m)[:k]) for k in p]).astype(np.int32)
    sel_w = g.uniform(0.05, 1.0, len(sel_idx))
    scale = 1.0 / np.sqrt(max(N - 1, 1))
    Sf, HSf = g.standard_normal((n, N)) * scale, g.standard_normal((m, N)) * scale
    xf, Hxf = g.standard_normal(n), g.standard_normal(m)
    yo = Hxf + g.standard_normal(m)
    sig2 = np.full(m, sigma * sigma)
    xa, Sa = loc_analysis_csr(zone_ptr, sel_ptr, sel_idx, sel_w, xf, Hxf, yo, Sf, HSf, sig2)[:2]
    xo, So = O.loc_analysis_csr(zone_ptr, sel_ptr, sel_idx, sel_w, xf, Hxf, yo, sig2, Sf, HSf)[:2]
    # rounding M by eps moves M^-1/2 and M^-1 by at most eps kappa (M >= I); N
    # sums of it in the products, both sides
    kappa = 1.0 + (HSf ** 2).sum() / sigma ** 2
    tol = 2 * max(N, 4) * np.finfo(float).eps * kappa
    assert rel_err(Sa, So) < tol
    # a = M^-1 b is compared through its increments, |b| / |a| <= kappa apart
    assert rel_err(xa - xf, xo - xf) < tol * max(1.0, np.abs(xf).max() / np.abs(xo - xf).max())
    np.testing.assert_array_equal(Sa[: zone_ptr[1]], Sf[: zone_ptr[1]])
    np.testing.assert_array_equal(xa[: zone_ptr[1]], xf[: zone_ptr[1]])

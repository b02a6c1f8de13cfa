"""Gram and update where an ensemble ends inside the last tile rows of its kernels,
on both sides of each tile row's end, for zones on both sides of the length at which
the observations are shared by four waves, against the oracle.  Needs an MI355X."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.kfcheck import rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [33, 48, 49, 80, 81, 96, 97, 112, 113, 128, 192, 193])
def test_padding_vs_oracle(N):
    from oak_amd.rrsqrt import loc_analysis_csr
    g = np.random.default_rng(1000 + N)
    p = np.array([1, 5, 130, 511, 0, 512, 701])
    m = int(p.max())
    zone_ptr = np.cumsum(np.r_[0, [1, 15, 16, 17, 3, 64, 65]])
    n = int(zone_ptr[-1])
    sel_ptr = np.r_[0, np.cumsum(p)]
    sel_idx = np.concatenate([np.sort(g.permutation(m)[:k]) for k in p]).astype(np.int32)
    sel_w = g.uniform(0.05, 1.0, len(sel_idx))
    scale = 1.0 / np.sqrt(N - 1)
    Sf, HSf = g.standard_normal((n, N)) * scale, g.standard_normal((m, N)) * scale
    xf, Hxf = g.standard_normal(n), g.standard_normal(m)
    yo = Hxf + g.standard_normal(m)
    sig2 = np.full(m, 0.25)
    xa, Sa = loc_analysis_csr(zone_ptr, sel_ptr, sel_idx, sel_w, xf, Hxf, yo, Sf, HSf, sig2)[:2]
    xo, So = O.loc_analysis_csr(zone_ptr, sel_ptr, sel_idx, sel_w, xf, Hxf, yo, sig2, Sf, HSf)[:2]
    # rounding M by eps moves M^-1/2 and M^-1 by at most eps kappa (M >= I); N
    # sums of it in the products, both sides
    kappa = 1.0 + (HSf ** 2).sum() / 0.25
    tol = 2 * N * np.finfo(float).eps * kappa
    assert rel_err(Sa, So) < tol
    # a = M^-1 b is compared through its increments, |b| / |a| <= kappa apart
    assert rel_err(xa - xf, xo - xf) < tol * max(1.0, np.abs(xf).max() / np.abs(xo - xf).max())
    z = slice(zone_ptr[4], zone_ptr[5])
    np.testing.assert_array_equal(Sa[z], Sf[z])
    np.testing.assert_array_equal(xa[z], xf[z])

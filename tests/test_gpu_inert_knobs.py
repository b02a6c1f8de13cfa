"""Settings that no longer choose anything are still taken, kept and without effect
on any bit of the analysis.  Needs an MI355X."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [24, 64, 100])
def test_no_effect(N):
    from oak_amd import assimilation as A
    from oak_amd import synth
    from oak_amd._lib import Context
    P = synth.column_ocean(20, 15, 2, N, 400, 60, seed_cfg=900 + N, hlen=4, vlen=1, L=3.0,
                           cutoff=9.0)
    H = A.coo_to_csr(P.m, P.Hi, P.Hj, P.Hs)
    geo = A.Geometry(P.zone_ptr, P.zpos, P.corr_len, P.max_len, P.ox, P.oy, metric=P.metric,
                     loctype=P.loctype)
    c = Context(0)
    ref = None
    for knobs in ({}, {"ql_zones": 4}, {"ql_zones": 32}, {"tri_split": 1}, {"tri_split": 4},
                  {"persist": 1}, {"persist": 2}):
        c.set_tuning(**knobs)
        assert all(c.tuning()[k] == v for k, v in knobs.items())
        Ea = A.ensemble_analysis(geo, H, P.Hshift, P.yo, P.rmse2, P.E, ctx=c)
        ref = Ea if ref is None else ref
        np.testing.assert_array_equal(Ea, ref)
    assert not np.array_equal(ref, P.E)
    c.close()

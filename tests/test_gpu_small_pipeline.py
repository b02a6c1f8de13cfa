"""Small ensembles on enough zones that their chunks run on several streams: the same
bits as in order on one stream, and as in many small chunks.  Needs an MI355X."""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,N", [(128, 128, 16), (97, 95, 32), (130, 129, 11), (97, 95, 29)])
def test_schedules_same_bits(nx, ny, N):
    from oak_amd import assimilation as A
    from oak_amd import synth
    from oak_amd._lib import Context
    P = synth.column_ocean(nx, ny, 1, N, 3000, 200, seed_cfg=700 + N, hlen=4, vlen=1, L=3.0,
                           cutoff=9.0)
    NP = 16 if N <= 16 else 32
    # run_zones: several streams from 4096 zones and 2^18 zones times rows on
    assert P.nzones >= 4096 and P.nzones * NP >= 1 << 18
    H = A.coo_to_csr(P.m, P.Hi, P.Hj, P.Hs)
    geo = A.Geometry(P.zone_ptr, P.zpos, P.corr_len, P.max_len, P.ox, P.oy, metric=P.metric,
                     loctype=P.loctype)
    out = []
    for timing, ws in ((False, None), (True, None), (False, 16 << 20)):
        if ws:
            os.environ["OAKG_WORKSPACE_BYTES"] = str(ws)
        try:
            c = Context(0)
        finally:
            os.environ.pop("OAKG_WORKSPACE_BYTES", None)
        c.set_timing(timing)
        slots = c.tuning()["slots"]
        # (the last chunk is a smaller one)
        assert slots > 1 and P.nzones % (64 * slots)
        for _ in range(2):  # the second with the streams' workspaces in place
            out.append(A.ensemble_analysis(geo, H, P.Hshift, P.yo, P.rmse2, P.E, inflation=1.02, ctx=c))
        c.close()
    for o in out[1:]:
        np.testing.assert_array_equal(out[0], o)
    assert not np.array_equal(out[0], P.E)

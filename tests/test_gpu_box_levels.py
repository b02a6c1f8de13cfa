"""Search levels of the observation operator on grids whose sides differ (boxes
that are points in some dimensions, grids of one cell, sides one above a power
of two) against the oracle's box tree: columns, weights and validity bit for
bit.  Needs an MI355X."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.test_gpu_obsoper import _curvilinear, _points

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(2,), (3,), (130,), (2, 2), (2, 33), (34, 3), (17, 2, 3),
                                   (2, 4, 18), (2, 2, 2, 2), (9, 2, 3, 2)])
def test_levels_bit_exact_vs_box_tree(shape):
    from oak_amd import assimilation as A
    g = np.random.default_rng(sum(shape))
    coords = _curvilinear(shape, seed=len(shape) + 1)
    m = 300
    pts = _points(coords, m, g, on_lines=0.4)
    obs_var = np.zeros(m, np.int32)
    grids = [dict(coords=coords, mask=g.uniform(size=shape) < 0.05)]
    got = A.obs_operator(grids, obs_var, list(pts))
    ref = O.obs_operator(grids, obs_var, list(pts))
    for a, b in zip(got, ref):
        np.testing.assert_array_equal(a, b)

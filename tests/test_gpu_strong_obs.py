"""M^-1/2 and M^1/2 1 where observations are precise: zones whose whole
ensemble space is strongly observed (every eigenvalue of M large), solved in
ensemble and in observation space, one near-exact observation, and the
likelihood.  References from the singular values of the scaled anomalies, which
never form M.  Needs an MI355X."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.kfcheck import rel_err

pytestmark = pytest.mark.gpu
EPS = np.finfo(float).eps


def _functions(St, dt):
    """T = M^-1/2 Omega, a = M^-1 b and the spectrum's range on the span of the
    rows of St, for M = I + St^T St, b = St^T dt."""
    N = St.shape[1]
    U, s, Vt = np.linalg.svd(St, full_matrices=False)
    mu, c = 1.0 + s * s, Vt @ np.ones(N)
    # (I - V V^T only where V is not square: its rounding would hide mu^-1/2)
    full = len(s) == N
    R = Vt.T @ (((1.0 / np.sqrt(mu) - (0.0 if full else 1.0)))[:, None] * Vt)
    v = Vt.T @ ((np.sqrt(mu) - (0.0 if full else 1.0)) * c)
    if not full:
        R, v = R + np.eye(N), v + np.ones(N)
    T = R @ O.rotate_vector(np.full(N, 1.0 / np.sqrt(N)), v / np.linalg.norm(v))
    return T, Vt.T @ (s / mu * (U.T @ dt)), mu[-1], mu[0]


def _zones(N, p, sigma, seed):
    """Zones of 2 rows; HSf of no particular structure (no zero row sums)."""
    g = np.random.default_rng(seed)
    p = np.asarray(p)
    m, nz = int(p.max()) + 5, len(p)
    zone_ptr = 2 * np.arange(nz + 1)
    sel_ptr = np.r_[0, np.cumsum(p)]
    sel_idx = np.concatenate([np.sort(g.permutation(m)[:k]) for k in p]).astype(np.int32)
    sel_w = g.uniform(0.5, 1.0, len(sel_idx))
    Sf, HSf = g.standard_normal((2 * nz, N)), g.standard_normal((m, N))
    xf, Hxf = g.standard_normal(2 * nz), g.standard_normal(m)
    yo = Hxf + g.standard_normal(m)
    return zone_ptr, sel_ptr, sel_idx, sel_w, xf, Hxf, yo, Sf, HSf, np.full(m, sigma * sigma)


def _check(N, p, sigma, ctx=None, mode="all"):
    from oak_amd.rrsqrt import loc_analysis_csr
    args = _zones(N, p, sigma, seed=N)
    zone_ptr, sel_ptr, sel_idx, sel_w, xf, Hxf, yo, Sf, HSf, sig2 = args
    xa, Sa = loc_analysis_csr(*args, ctx=ctx)[:2]
    for z in range(len(p)):
        i = sel_idx[sel_ptr[z]:sel_ptr[z + 1]]
        r = sel_w[sel_ptr[z]:sel_ptr[z + 1]] / sigma
        T, a, lo, hi = _functions(r[:, None] * HSf[i], r * (yo - Hxf)[i])
        rows = slice(zone_ptr[z], zone_ptr[z + 1])
        # rounding M (or I + G) by eps moves its functions by eps hi / lo; N sums
        # of it in the products
        tol = 8 * max(N, 4) * EPS * hi / lo
        assert tol < 1e-10
        assert rel_err(Sa[rows], Sf[rows] @ T) < tol, (N, sigma, z, hi)
        if mode == "all":
            # a solves the normal equations: (hi / lo)^1/2 more of the innovations
            assert rel_err(xa[rows] - xf[rows], Sf[rows] @ a) < tol * np.sqrt(hi / lo), (N, sigma, z)


@pytest.mark.parametrize("sigma", [1e-2, 1e-4, 1e-5, 1e-7, 1e-9, 1e-12, 1e-20])
@pytest.mark.parametrize("N", [1, 2, 8, 16, 17, 32, 33, 40, 64, 65, 100, 128, 129, 200, 256])
def test_every_eigenvalue_large(N, sigma):
    _check(N, [3 * N + 2, 4 * N + 3, 3 * N + 5], sigma)


@pytest.mark.parametrize("sigma", [1e-4, 1e-7, 1e-9, 1e-12])
@pytest.mark.parametrize("N", [80, 128])
def test_observation_space_zones(N, sigma):
    from oak_amd._lib import Context
    c = Context(0)
    c.set_tuning(dual=64)
    try:
        _check(N, [1, 2, 7, 16, 17], sigma, ctx=c, mode="Sa")
    finally:
        c.close()


@pytest.mark.parametrize("sigma", [1e-6, 1e-8, 1e-9, 1e-10])
@pytest.mark.parametrize("N", [4, 16, 24, 32, 48, 64, 80, 128, 160, 256])
def test_one_precise_observation(N, sigma):
    """The analysed spread of the observed variable itself: |s M^-1/2| = |s| / (1 +
    |s|^2 / sigma^2)^1/2, close to sigma.  (The mean of T's columns is free of the
    rotation: T T^T = M^-1.)"""
    from oak_amd.rrsqrt import loc_analysis_csr
    g = np.random.default_rng(N)
    HSf = g.standard_normal((3, N))
    HSf /= np.linalg.norm(HSf, axis=1)[:, None]
    xa, Sa = loc_analysis_csr([0, 1, 2, 3], [0, 1, 2, 3], np.arange(3, dtype=np.int32), np.ones(3),
                              np.zeros(3), np.zeros(3), np.ones(3), HSf, HSf,
                              np.full(3, sigma * sigma))[:2]
    ref = 1.0 / np.sqrt(1.0 + sigma ** -2)
    # s M^-1/2 is a difference of terms of size 1: eps N of them against sigma
    np.testing.assert_allclose(np.linalg.norm(Sa, axis=1), ref, rtol=4 * N * EPS / sigma)
    np.testing.assert_allclose(xa, 1.0, rtol=4 * N * EPS / sigma)


@pytest.mark.parametrize("sigma", [1e-3, 1e-5, 1e-7, 1e-9])
@pytest.mark.parametrize("N", [33, 65, 100, 128])
def test_likelihood(N, sigma):
    """J and dJ/dlog sigma, all zones with p > N observations; no innovations, so
    that the gradient is what |M^-1/2 s~|^2 leaves of 1."""
    from oak_amd import synth
    from oak_amd.nll import evaluate, problem_from_ensemble
    from tests.nll_ref import selection
    P = synth.config3(nx=4, N=N, m=3 * N, seed_cfg=N)
    prob = problem_from_ensemble(P)
    m, nz = 3 * N, P.nzones
    # anomalies of full rank on the ensemble space, zones that see nearly all
    # observations with weights of order 1
    g = np.random.default_rng(N)
    prob.HSf = np.asfortranarray(g.standard_normal((m, N)))
    prob.yo = np.array(prob.Hxf)
    L = 200.0
    J, gth, gLz, ga = evaluate(prob, np.full(m, sigma ** 2), np.full(nz, L), 1.0)
    Jr, gr, kap = 0.0, np.zeros(m), 1.0
    for idx, dist in selection(P, prob.HSf):
        if len(idx) == 0:
            continue
        w = np.exp(-(np.asarray(dist) / L) ** 2)
        r = w * w / sigma ** 2
        St = np.sqrt(r)[:, None] * prob.HSf[idx]
        U, s, Vt = np.linalg.svd(St, full_matrices=False)
        mu = 1.0 + s * s
        kap = max(kap, mu[0] / mu[-1])
        Jr += 0.5 * (np.log(mu).sum() - np.log(r).sum())
        gr[idx] += 1.0 - ((U * (s * s / mu)) * U).sum(axis=1)  # 1 - s~^T M^-1 s~
    tol = 64 * N * EPS * kap
    assert tol < 1e-7
    assert np.abs(gth - gr).max() <= tol * np.abs(gr).max()
    assert abs(J - Jr) <= tol * abs(Jr)

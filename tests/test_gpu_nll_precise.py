"""The likelihood where observations are precise: zones with fewer observations than
members, whose derivatives are what the observations leave of 1, and zones whose
M or innovation covariance has unit eigenvalues below its own rounding.
References from the singular values of the scaled anomalies, which never form M.
Needs an MI355X."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
EPS = np.finfo(float).eps


def _problem(N, counts):
    """Zones of one row, 1000 apart, counts[k] observations (weight 1) at zone k."""
    from oak_amd.assimilation import Geometry
    from oak_amd.nll import NLLProblem
    g = np.random.default_rng(N)
    nz, m = len(counts), sum(counts)
    zpos = np.zeros((nz, 4))
    zpos[:, 0] = 1000.0 * np.arange(nz)
    HS = np.asfortranarray(g.standard_normal((m, N)) / np.sqrt(N))
    geo = Geometry(np.arange(nz + 1), zpos, np.full(nz, 1e9), np.full(nz, 10.0),
                   np.repeat(zpos[:, 0], counts), np.zeros(m))
    return NLLProblem(geo, np.zeros(m), g.standard_normal(m), HS, N)


@pytest.mark.parametrize("sigma", [1e-4, 1e-5, 1e-7, 1e-9, 1e-11])
@pytest.mark.parametrize("N", [8, 16, 24, 32, 40, 64, 65, 90, 100, 128])
def test_likelihood(N, sigma):
    from oak_amd.nll import evaluate
    counts = [N // 8, N // 4, 1, 520, N // 6]
    prob = _problem(N, counts)
    J, gth, gL, ga = evaluate(prob, np.full(prob.m, sigma ** 2), np.full(len(counts), 1e9), 1.0)
    assert np.isfinite(gth).all() and np.isfinite(gL).all() and np.isfinite(ga)
    Jr, tolJ, k0 = 0.0, 0.0, 0
    for p in counts:
        rows = slice(k0, k0 + p)
        k0 += p
        dt = prob.yo[rows] / sigma
        U, s, _ = np.linalg.svd(prob.HSf[rows] / sigma, full_matrices=False)
        mu = 1.0 + s * s
        # (I + S~ S~^T)^-1 d~ and its diagonal, without differences where p <= N
        if p <= N:
            t, om = U @ (U.T @ dt / mu), ((U * U) / mu).sum(axis=1)
        else:
            t = dt - U @ (s * s / mu * (U.T @ dt))
            om = 1.0 - ((U * U) * (s * s / mu)).sum(axis=1)
        Jr += 0.5 * (dt @ t + np.log(mu).sum()) + p * np.log(sigma)
        # rounding moves D~ = I + S~ S~^T (p < N; M otherwise) by eps hi, so its inverse
        # by eps hi / lo of itself; sums over N and p
        c = 4 * max(N, p) * EPS * mu[0] / mu[-1]
        t2 = p * np.abs(t).max() ** 2
        assert np.abs(gth[rows] - (om - t * t)).max() <= c * (om.max() + 2 * t2), p
        tolJ += c * (dt @ t + p) + 1e-14 * abs(p * np.log(sigma))
    assert abs(J - Jr) <= tolJ


@pytest.mark.parametrize("sigma", [1e-8, 1e-10])
@pytest.mark.parametrize("N", [2, 8, 16, 24, 32, 64, 65, 100, 128])
def test_bounded_below_the_rounding(N, sigma):
    """Pairs of observations of the same state (p < N), and centred anomalies (p >= N):
    unit eigenvalues that rounding by eps sigma^-2 leaves anywhere."""
    from oak_amd.nll import evaluate
    counts = [2 * max(1, N // 5), 3 * N, 530]
    prob = _problem(N, counts)
    HS = prob.HSf
    HS -= HS.mean(axis=1, keepdims=True)
    HS[1:counts[0]:2] = HS[:counts[0]:2]
    J, gth, gL, ga = evaluate(prob, np.full(prob.m, sigma ** 2), np.full(len(counts), 1e9), 1.0)
    assert np.isfinite(J) and np.isfinite(ga) and np.isfinite(gL).all()
    # 0 <= r u <= 1 and |e~| <= |d~| for any positive definite D~ >= I
    dt2 = (prob.yo @ prob.yo) / sigma ** 2
    assert np.abs(gth).max() <= 2 * (1 + dt2)

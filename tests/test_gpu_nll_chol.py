"""The likelihood's kernel for N <= 64 at the ensemble sizes where its tiles end,
for zones with no, few and so many observations (700) that four waves share
them, against the dense FP64 reference (the long zones: extended precision).
Needs an MI355X."""
import numpy as np
import pytest
import torch

from tests.nll_ref import nll_reference, selection

pytestmark = pytest.mark.gpu


def _extended(sel, HSf, innov, log_sigma, L, a):
    """J and its derivatives from the ensemble-space formulas in extended
    precision.  (With 700 observations per zone the dense reference's p x p
    solve has a condition number of 2e7, and dJ/da, a difference of two large
    terms, loses seven digits in it.)"""
    ld = np.longdouble
    HS, innov = np.asarray(HSf, ld) * ld(a), np.asarray(innov, ld)
    s2 = np.exp(2 * np.asarray(log_sigma, ld))
    N = HS.shape[1]
    J, gL, ga, gth = ld(0), ld(0), ld(0), np.zeros(len(innov), ld)
    for idx, dist in sel:
        lw = -(np.asarray(dist, ld) / ld(L)) ** 2
        r, S, d = np.exp(2 * lw) / s2[idx], HS[idx], innov[idx]
        b = S.T @ (r * d)
        X = np.concatenate([np.eye(N, dtype=ld) + S.T @ (r[:, None] * S), b[:, None],
                            np.eye(N, dtype=ld)], axis=1)
        logdet = ld(0)
        for k in range(N):
            logdet += np.log(X[k, k])
            X[k] /= X[k, k]
            for i in range(N):
                if i != k:
                    X[i] -= X[i, k] * X[k]
        av, Mi = X[:, N], X[:, N + 1:]
        J += 0.5 * ((r * d * d).sum() - b @ av - np.log(r).sum() + logdet)
        g = 0.5 * ((d - S @ av) ** 2 + ((S @ Mi) * S).sum(axis=1) - 1 / r)
        gth[idx] -= 2 * r * g
        gL += (g * r * -4 * lw).sum() / ld(L)
        ga += (N - np.trace(Mi) - av @ av) / ld(a)
    return float(J), gth.astype(float), float(gL), float(ga)


@pytest.mark.parametrize("nx,m", [(10, 70), (40, 90), (6, 700)])
@pytest.mark.parametrize("N", [2, 16, 17, 32, 33, 48, 64])
def test_nll_vs_reference(N, nx, m):
    from oak_amd import synth
    from oak_amd.nll import evaluate, problem_from_ensemble
    P = synth.config3(nx=nx, N=N, m=m, seed_cfg=N)
    prob = problem_from_ensemble(P)
    nz = P.nzones
    ls = 0.5 * np.log(P.rmse2) - 0.4
    L, a = 3.5, 1.1
    J, gth, gLz, ga = evaluate(prob, np.exp(2 * ls), np.full(nz, L), a)
    sel = selection(P, prob.HSf)
    if m > 512:
        Jr, gthr, gLr, gar = _extended(sel, prob.HSf, prob.yo - prob.Hxf, ls, L, a)
    else:
        lsr = torch.as_tensor(ls).clone().requires_grad_(True)
        Lr = torch.tensor(L, dtype=torch.float64, requires_grad=True)
        ar = torch.tensor(a, dtype=torch.float64, requires_grad=True)
        Jt = nll_reference(sel, prob.HSf, prob.Hxf, prob.yo, lsr, Lr, ar)
        Jt.backward()
        Jr, gthr, gLr, gar = float(Jt.detach()), lsr.grad.numpy(), float(Lr.grad), float(ar.grad)
    # the bounds of the other likelihood tests (D^-1 of the reference loses
    # the ratio of its diagonal, w^-2 <= e^(2 (15 / 3.5)^2), to rounding)
    assert abs(J - Jr) <= 1e-9 * abs(Jr)
    assert np.abs(gth - gthr).max() <= 1e-8 * np.abs(gthr).max()
    assert abs(gLz.sum() - gLr) <= 1e-8 * max(1.0, abs(gLr))
    assert abs(ga - gar) <= 1e-8 * max(1.0, abs(gar))

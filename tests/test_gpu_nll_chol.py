"""The likelihood's kernel for N <= 64 at the ensemble sizes where its tiles end,
for zones with no, few and so many observations (700) that four waves share
them, against the dense FP64 reference.  Needs an MI355X."""
import numpy as np
import pytest
import torch

from tests.nll_ref import nll_reference, selection

pytestmark = pytest.mark.gpu


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
    lsr = torch.as_tensor(ls).clone().requires_grad_(True)
    Lr = torch.tensor(L, dtype=torch.float64, requires_grad=True)
    ar = torch.tensor(a, dtype=torch.float64, requires_grad=True)
    Jr = nll_reference(selection(P, prob.HSf), prob.HSf, prob.Hxf, prob.yo, lsr, Lr, ar)
    Jr.backward()
    # the bounds of the other likelihood tests (D^-1 of the reference loses
    # the ratio of its diagonal, w^-2 <= e^(2 (15 / 3.5)^2), to rounding)
    assert abs(J - float(Jr.detach())) <= 1e-9 * abs(float(Jr.detach()))
    gthr = lsr.grad.numpy()
    assert np.abs(gth - gthr).max() <= 1e-8 * np.abs(gthr).max()
    assert abs(gLz.sum() - float(Lr.grad)) <= 1e-8 * max(1.0, abs(float(Lr.grad)))
    assert abs(ga - float(ar.grad)) <= 1e-8 * max(1.0, abs(float(ar.grad)))

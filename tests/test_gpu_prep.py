"""Rows gathered and scattered at the ends of a workgroup's run, and H on the
members for rows of no to nine entries and member counts around a workgroup's
share, against numpy and the oracle.  Needs an MI355X."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests.kfcheck import rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("n,N", [(1, 1), (255, 3), (2048, 9), (2049, 2), (16385, 5), (40000, 33)])
def test_permute_rows(n, N, dtype):
    from oak_amd.layout import _permute
    g = torch.Generator().manual_seed(n)
    full = n + 13
    idx = torch.randperm(full, generator=g)[:n].cuda()
    src = torch.randn((N, full), generator=g, dtype=dtype).cuda().t()
    dst = torch.full((N, n), -1.0, dtype=dtype, device="cuda").t()
    _permute(True, idx, full, src, dst, None)
    assert torch.equal(dst, src[idx])
    back = torch.full((N, full), -2.0, dtype=dtype, device="cuda").t()
    _permute(False, idx, full, dst, back, None)
    ref = torch.full((full, N), -2.0, dtype=dtype, device="cuda")
    ref[idx] = dst
    assert torch.equal(back, ref)


def test_permute_rows_index_out_of_range():
    from oak_amd._lib import OakError
    from oak_amd.layout import _permute
    idx = torch.arange(3000).cuda()
    idx[2999] = 3000
    src = torch.zeros((2, 3000), dtype=torch.float64, device="cuda").t()
    dst = torch.zeros((2, 3000), dtype=torch.float64, device="cuda").t()
    with pytest.raises(OakError):
        _permute(True, idx, 3000, src, dst, None)


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("N", [2, 8, 9, 32, 33, 70])
def test_operator_on_members(N, fp32):
    from oak_amd.assimilation import ensemble_report
    g = np.random.default_rng(N)
    n, m = 500, 300
    cnt = g.integers(0, 10, m)
    cnt[:10] = np.arange(10)
    rp = np.r_[0, np.cumsum(cnt)].astype(np.int64)
    col = g.integers(0, n, rp[-1]).astype(np.int32)
    val = g.uniform(0.1, 1.0, rp[-1])
    E = np.asfortranarray(g.standard_normal((n, N)).astype(np.float32 if fp32 else np.float64))
    sh = np.zeros(m, E.dtype)
    yo, sig2 = g.standard_normal(m), np.full(m, 0.3)
    got = ensemble_report((rp, col, val), sh, yo, sig2, E, ranges=np.array([0, 10, m]))
    ref = O.ensemble_report((np.repeat(np.arange(m), cnt), col, val), sh.astype(float), yo, sig2,
                            E.astype(float), ranges=np.array([0, 10, m]))
    # FP32 members: HS is stored in FP32 (N terms a row), the rest in FP64
    assert rel_err(got, ref) < (N * 2.0 ** -23 if fp32 else 1e-12)

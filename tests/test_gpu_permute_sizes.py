"""Gathers and scatters of states so large that a workgroup takes several members
(from two on) and sorts its rows (from eight): bit for bit against torch
indexing.  Needs an MI355X."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

ROWS = 2048  # of a workgroup


def _members(n, N):
    """Members of a workgroup (launch_permute_rows)."""
    gx = -(-(-(-n // ROWS)) // 8) * 8
    groups = min(N, max(1, -(-4096 // gx)))
    return -(-N // groups)


def _indices(order, n, full_len, g):
    if order == "shuffled":
        return g.permutation(full_len)[:n]
    if order == "strided":  # columns of 30 levels, a slab apart
        slab = full_len // 30
        return (np.arange(slab)[:, None] + slab * np.arange(30)[None, :]).reshape(-1)[:n]
    idx = g.choice(full_len, n, replace=False)  # runs of 1..300 ascending, some reversed
    idx.sort()
    for a in range(0, n, 300):
        if g.uniform() < 0.3:
            idx[a:a + 300] = idx[a:a + 300][::-1]
    return idx


@pytest.mark.parametrize("order", ["shuffled", "strided", "runs"])
@pytest.mark.parametrize("dtype,n,N,members", [
    (torch.float32, 270_001, 250, 9),   # sorted; 7 members in the last group
    (torch.float64, 270_001, 250, 9),
    (torch.float32, 1_050_000, 61, 8),  # sorted; 5 in the last group
    (torch.float64, 60_001, 251, 2),    # not sorted, 1 in the last group
    (torch.float32, 100_001, 250, 4),
    (torch.float64, 220_001, 250, 7),
])
def test_gather_scatter(dtype, n, N, members, order):
    from oak_amd import layout as Lay
    assert _members(n, N) == members and n % ROWS and N % members
    g = np.random.default_rng(n + N)
    full_len = 30 * (n // 30 + 200)
    idx = _indices(order, n, full_len, g)
    assert len(idx) == n
    di = torch.as_tensor(idx, device="cuda:0")
    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(n)
    src = torch.randn((N, full_len), generator=gen, device="cuda:0", dtype=dtype).t()
    out = torch.full((N, n), -2.0, dtype=dtype, device="cuda:0").t()
    Lay._permute(True, idx, full_len, src, out, None)
    assert torch.equal(out.t(), src.t()[:, di])
    back = torch.full((N, full_len), -3.0, dtype=dtype, device="cuda:0").t()
    Lay._permute(False, idx, full_len, out, back, None)
    ref = torch.full((N, full_len), -3.0, dtype=dtype, device="cuda:0")
    ref[:, di] = out.t()
    assert torch.equal(back.t(), ref)
    # a gather may read an element twice
    idx[1::7] = idx[0]
    Lay._permute(True, idx, full_len, src, out, None)
    assert torch.equal(out.t(), src.t()[:, torch.as_tensor(idx, device="cuda:0")])


@pytest.mark.parametrize("bad", [-1, "past"])
@pytest.mark.parametrize("n,N", [(270_001, 250), (60_001, 251)])
def test_index_out_of_range(n, N, bad):
    """An argument error, and the other elements of the workgroup are stored."""
    from oak_amd import _lib
    from oak_amd import layout as Lay
    full_len = n + 999
    idx = np.random.default_rng(n).permutation(full_len)[:n]
    where = n - 5  # in the last run of rows
    idx[where] = full_len if bad == "past" else bad
    src = torch.arange(full_len, device="cuda:0", dtype=torch.float32).repeat(N, 1).t()
    out = torch.full((N, n), -2.0, dtype=torch.float32, device="cuda:0").t()
    with pytest.raises(_lib.OakError):
        Lay._permute(True, idx, full_len, src, out, None)
    keep = np.delete(np.arange(n), where)
    assert torch.equal(out.t()[:, torch.as_tensor(keep, device="cuda:0")],
                       torch.as_tensor(idx[keep], device="cuda:0").float().expand(N, -1))
    back = torch.full((N, full_len), -3.0, dtype=torch.float32, device="cuda:0").t()
    out.copy_(torch.arange(n, device="cuda:0", dtype=torch.float32)[:, None].expand(n, N))
    with pytest.raises(_lib.OakError):
        Lay._permute(False, idx, full_len, out, back, None)
    ref = torch.full((full_len,), -3.0, device="cuda:0")
    ref[torch.as_tensor(idx[keep], device="cuda:0")] = torch.as_tensor(keep, device="cuda:0").float()
    assert torch.equal(back.t(), ref.expand(N, -1))

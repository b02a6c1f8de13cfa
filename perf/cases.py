"""Workloads that a user of oak_amd runs, for timing and for comparing outputs.

Every case goes through the public entry points (``oak_amd.assimilation``,
``oak_amd.nll`` and the C ABI of include/oakg.h for the state layout).  The
cases are described by plain sizes:

* ``analysis`` / ``loc``: a model grid of nx x ny columns, each a zone holding
  ``vars`` variables on ``levels`` levels plus one surface variable, ``members``
  ensemble members, observations of the surface (``uniform``, along satellite
  ``tracks``, or in ``swaths`` whose local counts are roughly log-normal, with
  gaps without data) and ``profiles`` columns observed on every level;
  localisation length and cutoff in grid cells.  ``analysis`` is oak_assim's
  ensemble path (ensemble_analysis, FP64 or mixed precision), ``loc`` is
  locAnalysis on anomalies (loc_analysis).
* ``nll``: the innovation likelihood with its gradient, one step of the
  hyperparameter tuning.
* ``report``: the innovation statistics of an ensemble.
* ``operator``: the observation operator from grid coordinates (host arrays).
* ``fields``: members gathered into the zone-permuted state and scattered back
  (what loading and saving an ensemble does on the GPU).

Members are Gaussian random fields of unit variance, observations point values
of a truth member plus noise of the stated error; all from the seed.
"""
import ctypes
import math
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import torch

import oak_amd
from oak_amd import OAKG_FP64, OAKG_MIXED, autotune
from oak_amd.assimilation import (CARTESIAN, SPHERICAL, SPHERICAL_APPROX, Geometry,
                                  ensemble_analysis, ensemble_report, loc_analysis, obs_operator)
from oak_amd.nll import NLLProblem, innovation_nll
from oak_amd.rrsqrt import default_context

DEV = "cuda:0"
EARTH = 6378137.0
DEGREES = 0.25  # grid spacing of the longitude-latitude cases
METRIC = {"cartesian": CARTESIAN, "spherical": SPHERICAL, "approx": SPHERICAL_APPROX}


def _analysis(name, nx, ny, levels, vars, members, obs, surface, profiles, precision="fp64",
              metric="cartesian", op="analysis", L=6.0, cutoff=18.0, sigma=0.03, inflation=1.0,
              clamp=False):
    c = {"op": op, "nx": nx, "ny": ny, "levels": levels, "vars": vars, "members": members,
         "obs": obs, "surface": surface, "profiles": profiles, "precision": precision,
         "metric": metric, "L": L, "cutoff": cutoff, "sigma": sigma, "inflation": inflation,
         "clamp": clamp}
    return dict(c, name=name) if name else c


def listed():
    return [
        # a toy domain, as in the first steps with the library and in its
        # tests: launches and host work are all there is
        _analysis("grid8_n8", 8, 8, 1, 0, 8, "uniform", 20, 0, L=3.0, cutoff=6.0, sigma=0.1),
        # a 2-D field with one zone per point (benchmark configuration 0)
        _analysis("grid64_n16", 64, 64, 1, 0, 16, "uniform", 400, 0, L=5.0, cutoff=15.0,
                  sigma=0.1),
        # one step of hyperparameter tuning (benchmark configuration 3)
        {"name": "nll_256_n32", "op": "nll", "nx": 256, "ny": 256, "members": 32, "surface": 4000,
         "L": 2.5, "cutoff": 15.0},
        # a regional model with an ensemble size that fills no tile, some of
        # its inflation and the clamp of the corrections in use
        _analysis("coast_n40", 90, 61, 15, 4, 40, "tracks", 8000, 60, inflation=1.05, clamp=True),
        # a basin with track altimetry and profiles (benchmark configuration 1)
        _analysis("ocean_n64", 360, 180, 30, 4, 64, "tracks", 150000, 1700),
        # locAnalysis on longitude and latitude (great-circle distances)
        _analysis("lonlat_n100", 96, 60, 10, 4, 100, "swaths", 150, 20, op="loc",
                  metric="spherical"),
        # the headline workload in both precisions (benchmark configuration 2)
        _analysis("ocean_n128_mixed", 360, 180, 30, 4, 128, "swaths", 150, 60, precision="mixed"),
        _analysis("ocean_n128_fp64", 360, 180, 30, 4, 128, "swaths", 150, 60),
        # the largest ensembles on a sixteenth of benchmark configuration 4
        _analysis("ocean_n256_mixed", 180, 90, 40, 4, 256, "swaths", 1900, 625,
                  precision="mixed", L=3.0, cutoff=9.0),
        # the statistics written to the log before and after each analysis
        {"name": "report_n100", "op": "report", "nx": 180, "ny": 90, "levels": 30, "vars": 1,
         "members": 100, "surface": 150000, "profiles": 1700, "precision": "mixed"},
        # the operator of a cycle's observations on a 3-D grid with land
        {"name": "operator_3d", "op": "operator", "nx": 120, "ny": 90, "levels": 20,
         "observations": 40000},
        # a 4-variable state of config 1's grid with a third of land points
        {"name": "fields_n32", "op": "fields", "nodes": 7840800, "members": 32,
         "precision": "fp64"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.random()
    if kind < 0.08:
        nx = _log(rng, 16, 256)
        return {"op": "nll", "nx": nx, "ny": max(8, int(nx * rng.uniform(0.4, 1.0))),
                "members": _log(rng, 4, 64), "surface": _log(rng, 50, 4000),
                "L": round(rng.uniform(2.0, 6.0), 2), "cutoff": 15.0}
    if kind < 0.16:
        return {"op": "report", "nx": _log(rng, 20, 180), "ny": _log(rng, 20, 90),
                "levels": _log(rng, 1, 30), "vars": 1, "members": _log(rng, 4, 256),
                "surface": _log(rng, 200, 150000), "profiles": _log(rng, 1, 1700),
                "precision": rng.choice(["fp64", "mixed"])}
    if kind < 0.22:
        return {"op": "operator", "nx": _log(rng, 8, 120), "ny": _log(rng, 8, 90),
                "levels": _log(rng, 3, 20), "observations": _log(rng, 100, 40000)}
    if kind < 0.28:
        return {"op": "fields", "nodes": _log(rng, 3000, 7000000), "members": _log(rng, 3, 32),
                "precision": rng.choice(["fp64", "mixed"])}
    N = _log(rng, 4, 256)
    # zones up to what costs no more than the largest listed cases
    zmax = min(64800, int(9e11 / (max(N, 24) ** 3 + 2e5)), int(4e8 / N))
    zones = _log(rng, 64, zmax)
    nx = max(8, int(math.sqrt(zones * rng.uniform(0.8, 2.5))))
    ny = max(8, zones // nx)
    levels, vars_ = _log(rng, 1, 40), rng.randint(0, 4)
    while nx * ny * (levels * vars_ + 1) * N > 1.0e9:
        levels, vars_ = max(1, levels // 2), max(1, vars_ - 1)
    L = rng.choice([3.0, 5.0, 6.0])
    obs = rng.choice(["uniform", "tracks", "swaths"])
    if obs == "swaths":
        surface = _log(rng, 30, 600)  # median local count
    else:
        # mean local counts from a handful to two thousand
        surface = max(5, int(_log(rng, 8, 2000) * nx * ny / (math.pi * 9 * L * L)))
    metric = rng.choice(["cartesian"] * 4 + ["spherical", "approx"])
    if metric != "cartesian":
        per_zone = nx * ny / (math.pi * 9 * L * L) if obs == "swaths" else 1.0
        surface = max(5, min(surface, int(6e8 / (nx * ny) / per_zone)))
    return _analysis(None, nx, ny, levels, vars_, N, obs, surface,
                     _log(rng, 1, max(2, nx * ny // 100)) if vars_ else 0,
                     precision=rng.choice(["fp64", "mixed"]) if metric == "cartesian" else "fp64",
                     metric=metric, op="analysis" if metric == "cartesian" else
                     rng.choice(["analysis", "loc"]), L=L, cutoff=3 * L,
                     sigma=rng.choice([0.03, 0.1]),
                     inflation=rng.choice([1.0, 1.0, 1.05, 1.2]), clamp=rng.random() < 0.25)


# --------------------------------------------------------------------------
# inputs
# --------------------------------------------------------------------------
def _smoother(n, length, dev, dtype):
    """Rows of a Gaussian filter that gives unit-variance fields with
    correlation exp(-(r / length)^2) from white noise."""
    i = torch.arange(n, device=dev, dtype=torch.float64)
    k = torch.exp(-2.0 * ((i[:, None] - i[None, :]) / length) ** 2)
    return (k / k.square().sum(1, keepdim=True).sqrt()).to(dtype)


def _members(gen, nx, ny, levels, nvar, count, dtype):
    """``count`` members, one row of nx * ny * (nvar * levels + 1) values each,
    column by column (x fastest): the variables level by level, the surface."""
    kx = _smoother(nx, 10.0 if nx > 64 else 8.0, DEV, dtype)
    ky = _smoother(ny, 10.0 if ny > 64 else 8.0, DEV, dtype)
    kz = _smoother(levels, 5.0, DEV, dtype)
    s = nvar * levels + 1
    out = torch.empty((count, nx * ny * s), dtype=dtype, device=DEV)
    step = max(1, min(count, int(2e7 / (nx * ny * s))))
    for k in range(0, count, step):
        b = min(step, count - k)
        rows = out[k:k + b].view(b, ny, nx, s)
        if nvar:
            w = torch.randn((b * nvar * ny, nx, levels), generator=gen, device=DEV, dtype=dtype)
            w = (w.reshape(-1, levels) @ kz.t()).view(b, nvar, ny, nx, levels)
            w = (w.permute(0, 1, 2, 4, 3).reshape(-1, nx) @ kx.t()).view(b, nvar, ny, levels, nx)
            w = (w.permute(0, 1, 3, 4, 2).reshape(-1, ny) @ ky.t()).view(b, nvar, levels, nx, ny)
            rows[..., :s - 1] = w.permute(0, 4, 3, 1, 2).reshape(b, ny, nx, s - 1)
        w = torch.randn((b * ny, nx), generator=gen, device=DEV, dtype=dtype) @ kx.t()
        w = w.view(b, ny, nx).permute(0, 2, 1).reshape(-1, ny) @ ky.t()
        rows[..., s - 1] = w.view(b, nx, ny).permute(0, 2, 1)
    return out


def _surface_positions(g, c):
    """Observation positions in cell coordinates 1 .. nx, 1 .. ny."""
    nx, ny, how = c["nx"], c["ny"], c.get("obs", "tracks")
    if how == "uniform":
        return g.uniform(1, nx, c["surface"]), g.uniform(1, ny, c["surface"])
    if how == "tracks":
        want, xs, ys, have = c["surface"], [], [], 0
        per = min(1000, max(20, 2 * max(nx, ny)))
        while have < want:
            x0, y0, a = g.uniform(1, nx), g.uniform(1, ny), g.uniform(0, np.pi)
            t = np.linspace(-1.5, 1.5, per) * max(nx, ny)
            x, y = x0 + t * np.cos(a), y0 + t * np.sin(a)
            ok = (x >= 1) & (x < nx) & (y >= 1) & (y < ny)
            xs.append(x[ok])
            ys.append(y[ok])
            have += int(ok.sum())
        return np.concatenate(xs)[:want], np.concatenate(ys)[:want]
    smooth = lambda l: (_smoother(ny, l, "cpu", torch.float64).numpy() @ g.standard_normal((ny, nx))
                        @ _smoother(nx, l, "cpu", torch.float64).numpy().T)
    f, gap = smooth(50.0), smooth(40.0)
    f = (f - f.mean()) / max(f.std(), 0.1)
    spread = 0.97 if c["surface"] < 1000 else 0.45
    dens = c["surface"] / (math.pi * c["cutoff"] ** 2) * np.exp(spread * np.clip(f, -3.0, 2.6))
    cnt = g.poisson(dens * (gap > np.quantile(gap, 0.1)))
    jj, ii = np.nonzero(cnt)
    rep = cnt[jj, ii]
    x = np.repeat(ii + 1.0, rep) + g.uniform(0, 1, rep.sum())
    y = np.repeat(jj + 1.0, rep) + g.uniform(0, 1, rep.sum())
    ok = (x < nx) & (y < ny)
    return x[ok], y[ok]


def _observations(g, c, s):
    """Positions, errors and the operator H (4 entries a row) of the surface
    and profile observations, as numpy arrays."""
    nx, ny, levels = c["nx"], c["ny"], c.get("levels", 1)
    sx, sy = _surface_positions(g, c)
    np_ = c.get("profiles", 0)
    px, py = g.uniform(1, nx, np_), g.uniform(1, ny, np_)

    def corners(x, y):
        i = np.clip(np.floor(x).astype(np.int64), 1, nx - 1)
        j = np.clip(np.floor(y).astype(np.int64), 1, ny - 1)
        a, b = x - i, y - j
        w = np.stack([(1 - a) * (1 - b), a * (1 - b), (1 - a) * b, a * b], 1)
        z = np.stack([(i + di - 1) + nx * (j + dj - 1) for di, dj in
                      ((0, 0), (1, 0), (0, 1), (1, 1))], 1)
        return z, w

    z, w = corners(sx, sy)
    col, val = [(z * s + s - 1).ravel()], [w.ravel()]
    z, w = corners(px, py)
    lev = np.arange(levels)
    col.append((z[:, None, :] * s + lev[None, :, None]).ravel())
    val.append(np.repeat(w[:, None, :], levels, axis=1).ravel())
    x = np.concatenate([sx, np.repeat(px, levels)])
    y = np.concatenate([sy, np.repeat(py, levels)])
    sigma = np.concatenate([np.full(len(sx), c.get("sigma", 0.03)), np.full(np_ * levels, 0.5)])
    return x, y, sigma, np.concatenate(col).astype(np.int32), np.concatenate(val), len(sx)


def _dev(a, dtype=torch.float64):
    return torch.as_tensor(np.ascontiguousarray(a)).to(DEV, dtype)


def _world(c, seed):
    """Geometry, observations, operator and members of the gridded cases."""
    g = np.random.default_rng(seed)
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed)
    nx, ny, levels, nvar, N = c["nx"], c["ny"], c.get("levels", 1), c.get("vars", 0), c["members"]
    s = nvar * levels + 1
    x, y, sigma, col, val, nsurf = _observations(g, c, s)
    m, nz = len(x), nx * ny
    dtype = torch.float32 if c.get("precision") == "mixed" else torch.float64
    E = _members(gen, nx, ny, levels, nvar, N + 1, dtype)
    col_d, val_d = _dev(col, torch.int32), _dev(val)
    truth = (E[N][col_d.long()].double() * val_d).view(m, 4).sum(1)
    sig = _dev(sigma)
    yo = truth + sig * _dev(g.standard_normal(m))
    ii = np.tile(np.arange(1, nx + 1, dtype=float), ny)
    jj = np.repeat(np.arange(1, ny + 1, dtype=float), nx)
    scale = 1.0
    if c.get("metric", "cartesian") != "cartesian":
        # degrees; lengths in metres
        place = lambda a, a0: a0 + DEGREES * a
        x, y, ii, jj = place(x, -20.0), place(y, 30.0), place(ii, -20.0), place(jj, 30.0)
        scale = DEGREES * math.pi * EARTH / 180.0
    zpos = np.zeros((nz, 4))
    zpos[:, 0], zpos[:, 1] = ii, jj
    geo = Geometry(torch.arange(nz + 1, device=DEV, dtype=torch.int64) * s, _dev(zpos),
                   torch.full((nz,), c.get("L", 6.0) * scale, dtype=torch.float64, device=DEV),
                   torch.full((nz,), c.get("cutoff", 18.0) * scale, dtype=torch.float64,
                              device=DEV), _dev(x), _dev(y),
                   metric=METRIC[c.get("metric", "cartesian")])
    H = (torch.arange(m + 1, device=DEV, dtype=torch.int64) * 4, col_d, val_d)
    return {"geo": geo, "H": H, "yo": yo, "rmse2": sig * sig, "E": E[:N].t(), "m": m, "N": N,
            "surface": nsurf, "shift": torch.zeros(m, dtype=torch.float64, device=DEV)}


def _anomalies(w):
    """Mean and scaled anomalies of the members and of the observed members."""
    N, E = w["N"], w["E"]
    xf = E.mean(1)
    Sf = ((E - xf[:, None]).t().contiguous() / math.sqrt(N - 1.0)).t()
    return xf, Sf, *_observed(w)


def _observed(w):
    N, m = w["N"], w["m"]
    HE = torch.empty((N, m), dtype=torch.float64, device=DEV)
    col = w["H"][1].long()
    for k in range(N):
        HE[k] = (w["E"][:, k][col].double() * w["H"][2]).view(m, 4).sum(1)
    Hxf = HE.mean(0)
    return Hxf, ((HE - Hxf) / math.sqrt(N - 1.0)).t()


def _context(c):
    """The handle a program keeps, with the launch settings of the shipped
    table."""
    mixed = c.get("precision") == "mixed"
    ctx = default_context(0, OAKG_MIXED if mixed else OAKG_FP64)
    autotune.apply(ctx, c["members"], ctx.precision)
    return ctx


def _operator_inputs(c, seed):
    """A rectilinear 3-D grid with stretched levels and land, and the surface
    variable's 2-D grid; observations of both, a few outside the domain."""
    g = np.random.default_rng(seed)
    nx, ny, nl, m = c["nx"], c["ny"], c["levels"], c["observations"]
    ax = [np.cumsum(g.uniform(0.8, 1.2, nx)), np.cumsum(g.uniform(0.8, 1.2, ny)),
          np.cumsum(np.linspace(1.0, 4.0, nl))]
    land = np.zeros(nx * ny, bool)
    land[g.permutation(nx * ny)[:nx * ny // 30]] = True
    land = land.reshape(nx, ny)
    dry = land[:-1, :-1] | land[1:, :-1] | land[:-1, 1:] | land[1:, 1:]
    grids, used = [], 0
    for n in (3, 2):
        shape = (nx, ny, nl)[:n]
        mask = np.broadcast_to(land[:, :, None], shape) if n == 3 else land
        state = np.full(shape, -1, np.int64)
        sea = ~mask.ravel(order="F")
        flat = np.full(sea.size, -1, np.int64)
        flat[sea] = used + g.permutation(int(sea.sum()))
        used += int(sea.sum())
        state = flat.reshape(shape, order="F")
        coords = [np.asfortranarray(np.broadcast_to(
            ax[d].reshape([-1 if e == d else 1 for e in range(n)]), shape)) for d in range(n)]
        grids.append({"coords": coords, "mask": np.asfortranarray(mask), "state": state})
    # as many of each variable, and as many on land or outside, for every seed
    var = (np.arange(m) // 25 % 4 // 2).astype(np.int32)
    wet, shore = np.argwhere(~dry), np.argwhere(dry)
    cell = wet[g.integers(0, len(wet), m)]
    if len(shore):
        cell[::50] = shore[g.integers(0, len(shore), len(cell[::50]))]
    cell = np.column_stack([cell, g.integers(0, nl - 1, m)])
    pos = [a[i] + g.uniform(0.001, 0.999, m) * (a[i + 1] - a[i]) for a, i in zip(ax, cell.T)]
    pos[0][25::50] += ax[0][-1] - ax[0][0] + 1.0
    return grids, var, pos, ax


def _limit(c):
    """The clamp of the corrections per element of a column, or None."""
    if not c["clamp"]:
        return None
    lim = torch.full((c["vars"] * c["levels"] + 1,), 1.0, dtype=torch.float64, device=DEV)
    lim[-1] = 0.3
    return lim


def prepare(case, seed):
    c, op = case, case["op"]
    if op == "operator":
        grids, var, pos, _ = _operator_inputs(c, seed)
        return {"op": op, "grids": grids, "var": var, "pos": pos, "ctx": default_context()}
    if op == "fields":
        gen = torch.Generator(device=DEV)
        gen.manual_seed(seed)
        full, N = c["nodes"], c["members"]
        dtype = torch.float32 if c["precision"] == "mixed" else torch.float64
        # sea points in zone order: columns of a few levels lie together, the
        # levels a horizontal slab apart in the model's arrays
        levels = max(1, min(30, full // 64))
        slab = full // levels
        idx = (torch.arange(slab, device=DEV)[:, None]
               + slab * torch.arange(levels, device=DEV)[None, :])
        sea = torch.randperm(slab, generator=gen, device=DEV)[:max(1, int(0.67 * slab))]
        idx = idx[sea.sort().values].reshape(-1).contiguous()
        n = idx.numel()
        files = torch.randn((N, full), generator=gen, device=DEV, dtype=dtype)
        out = torch.full((N, full), 9999.0, dtype=dtype, device=DEV)
        return {"op": op, "idx": idx, "n": n, "full": full, "N": N, "files": files, "out": out,
                "state": torch.empty((N, n), dtype=dtype, device=DEV), "ctx": default_context()}
    if op == "nll":
        w = _world(dict(c, obs="uniform", sigma=0.1), seed)
        Hxf, HSf = _observed(w)
        prob = NLLProblem(w["geo"], Hxf, w["yo"], HSf.t().contiguous().t(), w["N"])
        return {"op": op, "prob": prob, "ctx": default_context(),
                "log_sigma": torch.full((w["m"],), math.log(0.3), dtype=torch.float64, device=DEV),
                "log_L": torch.tensor(math.log(c["L"]), dtype=torch.float64, device=DEV),
                "log_infl": torch.tensor(0.0, dtype=torch.float64, device=DEV)}
    w = _world(c, seed)
    if op == "report":
        return {"op": op, "w": w, "ranges": [0, w["surface"], w["m"]],
                "ctx": default_context(0, OAKG_MIXED if c["precision"] == "mixed" else OAKG_FP64)}
    state = {"op": op, "w": w, "ctx": _context(c), "inflation": c["inflation"]}
    if op == "loc":
        state["anomalies"] = _anomalies(w)
        return state
    # OAK's per-variable limit of the corrections, one value per element
    lim = _limit(c)
    state["limit"] = float("inf") if lim is None else lim.repeat(c["nx"] * c["ny"]).contiguous()
    state["out"] = torch.empty_like(w["E"].t()).t()
    return state


def run(state):
    op, ctx = state["op"], state["ctx"]
    if op == "operator":
        return obs_operator(state["grids"], state["var"], state["pos"], ctx=ctx)
    if op == "fields":
        lib = oak_amd.load()
        p = lambda t: ctypes.c_void_p(t.data_ptr())
        n, full, N, elem = state["n"], state["full"], state["N"], state["files"].element_size()
        ctx.check(lib.oakg_gather_rows(ctx.handle, n, N, p(state["idx"]), full, p(state["files"]),
                                       full, p(state["state"]), n, elem,
                                       oak_amd.OAKG_DEVICE_PTRS))
        ctx.check(lib.oakg_scatter_rows(ctx.handle, n, N, p(state["idx"]), full,
                                        p(state["state"]), n, p(state["out"]), full, elem,
                                        oak_amd.OAKG_DEVICE_PTRS))
        return state["state"], state["out"]
    if op == "nll":
        par = [state[k].clone().requires_grad_() for k in ("log_sigma", "log_L", "log_infl")]
        J = innovation_nll(*par, state["prob"], ctx)
        J.backward()
        return [J.detach()] + [p.grad for p in par]
    w = state["w"]
    if op == "report":
        return ensemble_report(w["H"], w["shift"], w["yo"], w["rmse2"], w["E"],
                               ranges=state["ranges"], ctx=ctx)
    if op == "loc":
        xf, Sf, Hxf, HSf = state["anomalies"]
        return loc_analysis(w["geo"], xf, Hxf, w["yo"], Sf, HSf, w["rmse2"], ctx=ctx)
    return ensemble_analysis(w["geo"], w["H"], w["shift"], w["yo"], w["rmse2"], w["E"],
                             inflation=state["inflation"], max_correction=state["limit"], ctx=ctx,
                             out=state["out"])


def work(case):
    """Each input read once and each output written once; the operations of
    the symmetric products, the eigensolve's 9 N^3, the transform and the
    update (for swaths the local counts are taken at their median)."""
    c, op = case, case["op"]
    if op == "operator":
        nodes = c["nx"] * c["ny"] * (c["levels"] + 1)
        return {"bytes": nodes * (3 * 8 + 9) + c["observations"] * (28 + 8 + 6 * 12), "flops": 0}
    if op == "fields":
        b = 4 if c["precision"] == "mixed" else 8
        n = int(0.67 * c["nodes"])
        return {"bytes": n * (16 + 4 * b * c["members"]), "flops": 0}
    N, nz = c["members"], c["nx"] * c["ny"]
    s = c.get("vars", 0) * c.get("levels", 1) + 1
    b = 4 if c.get("precision") == "mixed" else 8
    prof = c.get("profiles", 0) * c.get("levels", 1)
    disc = math.pi * c.get("cutoff", 18.0) ** 2 / nz
    if c.get("obs") == "swaths":
        p, m = c["surface"] + prof * disc, c["surface"] / disc + prof
    else:
        m = c["surface"] + prof
        p = m * min(1.0, disc)
    if op == "report":
        return {"bytes": m * (4 * b * N + 4 * 12 + 24), "flops": m * N * 12.0}
    flops = nz * (N * (N + 1) * p + 2 * N * p + 9.0 * N ** 3)
    if op == "nll":
        return {"bytes": 8 * m * (N + 4) + 8 * nz * 8, "flops": flops + nz * p * 2.0 * N * (N + 2)}
    flops += nz * (N ** 3 + 11.0 * N * N + 2.0 * s * N * (N + 1))
    return {"bytes": 2 * b * nz * s * N + m * (b * N + 80) + nz * 56, "flops": flops}


# --------------------------------------------------------------------------
# the same in 64 bits, by plain torch and numpy
# --------------------------------------------------------------------------
def _weights(geo, z0, z1, length):
    """Taper weights (zones x observations, 0 beyond the cutoff) and the
    distances."""
    zx, zy = geo.zpos[z0:z1, 0][:, None], geo.zpos[z0:z1, 1][:, None]
    if geo.metric == CARTESIAN:
        d = ((zx - geo.ox) ** 2 + (zy - geo.oy) ** 2).sqrt()
    elif geo.metric == SPHERICAL_APPROX:
        k = math.pi * EARTH / 180.0
        d = ((k * torch.cos((geo.oy + zy) * (math.pi / 360.0)) * (zx - geo.ox)) ** 2
             + (k * (zy - geo.oy)) ** 2).sqrt()
    else:
        r = math.pi / 180.0
        a, b = geo.oy * r, zy * r
        q = torch.sin(a) * torch.sin(b) + torch.cos(a) * torch.cos(b) * torch.cos((zx - geo.ox) * r)
        d = EARTH * torch.acos(q.clamp(-1.0, 1.0))
    w = torch.exp(-(d / length) ** 2)
    return torch.where(d <= geo.max_len[z0:z1][:, None], w, torch.zeros_like(w)), d


def _chunks(nz, m, N):
    step = max(1, int(2.5e9 / (8 * max(1, m) + 8 * 6 * N * N)))
    return [(k, min(nz, k + step)) for k in range(0, nz, step)]


def _rows_product(r, HS):
    """sum_l r[z, l] HS[l, i] HS[l, j] for each zone."""
    m, N = HS.shape
    out = torch.zeros((r.shape[0], N * N), dtype=torch.float64, device=DEV)
    step = max(1, int(2.5e9 / (8 * N * N)))
    for k in range(0, m, step):
        h = HS[k:k + step]
        out += r[:, k:k + step].contiguous() @ (h[:, :, None] * h[:, None, :]).reshape(-1, N * N)
    return out.view(-1, N, N)


def _eigh(M):
    """Batched eigendecomposition by LAPACK, the batch over threads."""
    host = M.cpu()
    parts = [p for p in host.split(max(1, -(-len(host) // 64)))]

    def solve(p):
        torch.set_num_threads(1)
        return torch.linalg.eigh(p)

    with ThreadPoolExecutor(8) as pool:
        got = list(pool.map(solve, parts))
    return torch.cat([a for a, _ in got]).to(DEV), torch.cat([b for _, b in got]).to(DEV)


def _perp(v):
    """Orthonormal basis of the complement of each v (zones x N), OAK's
    perpSpace."""
    N = v.shape[1]
    alpha = -1.0 / (v[:, -1].abs() + 1.0)
    sign = torch.where(v[:, -1] >= 0, 1.0, -1.0)
    u = v.clone()
    u[:, -1] += sign
    P = alpha[:, None, None] * u[:, :, None] * v[:, None, :N - 1]
    P[:, :N - 1, :] += torch.eye(N - 1, dtype=v.dtype, device=v.device)
    return P


def _transforms(w, Hxf, HSf, z0, z1):
    """The weights of the mean and the transform of the anomalies per zone,
    and which zones have observations."""
    N = w["N"]
    wt, _ = _weights(w["geo"], z0, z1, w["geo"].corr_len[z0:z1][:, None])
    r = wt * wt / w["rmse2"]
    C = _rows_product(r, HSf)
    rhs = (r * (w["yo"] - Hxf)) @ HSf
    lam, U = _eigh(C)
    mu = 1.0 + lam.clamp(min=0.0)
    Ut = U.transpose(1, 2).contiguous()
    a = torch.bmm(U, torch.bmm(Ut, rhs[:, :, None]) / mu[:, :, None])[:, :, 0]
    v = torch.bmm(U, Ut.sum(2, keepdim=True) * mu.sqrt()[:, :, None])[:, :, 0]
    v = v / v.norm(dim=1, keepdim=True)
    one = torch.full_like(v, 1.0 / math.sqrt(N))
    omega = v[:, :, None] * one[:, None, :]
    if N > 1:
        omega = omega + torch.bmm(_perp(v), _perp(one).transpose(1, 2).contiguous())
    T = torch.bmm(U, torch.bmm(Ut, omega) / mu.sqrt()[:, :, None])
    return a, T, (wt > 0).any(1)


def _exact_analysis(c, seed):
    nz, N = c["nx"] * c["ny"], c["members"]
    if nz * (N + 8.0) ** 3 > 2.6e10 or N < 2:
        return None
    w = _world(c, seed)
    if 3e-14 * w["m"] * nz * N * N > 8:
        return None
    E = w["E"]
    s = c["vars"] * c["levels"] + 1
    if c["op"] == "loc":
        xf, Sf, Hxf, HSf = _anomalies(w)
    else:
        Hxf, HSf = _observed(w)
        xf = E.t().mean(0, dtype=torch.float64)
    out = torch.empty((N, nz * s), dtype=torch.float64, device=DEV)
    xa = xf.clone()
    limit = _limit(c)
    for z0, z1 in _chunks(nz, w["m"], N):
        a, T, has = _transforms(w, Hxf, HSf, z0, z1)
        rows = slice(z0 * s, z1 * s)
        if c["op"] == "loc":
            S = Sf[rows].contiguous()
        else:
            S = (E[rows].double() - xf[rows, None]) / math.sqrt(N - 1.0)
        S = S.reshape(z1 - z0, s, N)
        inc = torch.bmm(S, a[:, :, None])[:, :, 0]
        Sa = torch.where(has[:, None, None], torch.bmm(S, T), S)
        if c["op"] == "loc":
            out[:, rows] = Sa.reshape(-1, N).t()
            xa[rows] += inc.reshape(-1)
            continue
        if limit is not None:
            inc = torch.minimum(torch.maximum(inc, -limit), limit)
        new = xf[rows] + inc.reshape(-1)
        Sa = c["inflation"] * math.sqrt(N - 1.0) * Sa
        out[:, rows] = new + Sa.reshape(-1, N).t()
    return (xa, out.t()) if c["op"] == "loc" else out.t()


def _exact_nll(c, seed):
    state = prepare(c, seed)
    prob, N, m, nz = state["prob"], c["members"], c["surface"], c["nx"] * c["ny"]
    if 3e-14 * m * nz * N * N > 8:
        return None
    S, d = prob.HSf, prob.yo - prob.Hxf
    sig2 = torch.exp(2.0 * state["log_sigma"])
    L = math.exp(float(state["log_L"]))
    J = torch.zeros((), dtype=torch.float64, device=DEV)
    gs = torch.zeros(m, dtype=torch.float64, device=DEV)
    gL, ga = J.clone(), J.clone()
    outer = (S[:, :, None] * S[:, None, :]).reshape(m, N * N)
    eye = torch.eye(N, dtype=torch.float64, device=DEV)
    for z0, z1 in _chunks(nz, 4 * m, N):
        w, dist = _weights(prob.geo, z0, z1, L)
        on = w > 0
        r = w * w / sig2
        M = (r @ outer).view(-1, N, N) + eye
        F = torch.linalg.cholesky(M)
        Minv = torch.cholesky_inverse(F)
        b = (r * d) @ S
        a = torch.bmm(Minv, b[:, :, None])[:, :, 0]
        t = a @ S.t()
        q = Minv.reshape(-1, N * N) @ outer.t()
        log_r = torch.where(on, torch.log(torch.where(on, r, torch.ones_like(r))), 0.0)
        logdet = 2.0 * torch.diagonal(F, dim1=1, dim2=2).log().sum(1)
        J += 0.5 * ((r * d * d).sum() - (b * a).sum() - log_r.sum() + logdet.sum())
        dr = torch.where(on, 0.5 * r * ((d - t) ** 2 + q) - 0.5, 0.0)  # r dJ/dr
        gs += -2.0 * dr.sum(0)
        gL += (dr * 4.0 * dist * dist / L ** 2).sum()
        ga += (N - torch.diagonal(Minv, dim1=1, dim2=2).sum(1) - (a * a).sum(1)).sum()
    return [J, gs, gL, ga]


def _exact_report(c, seed):
    w = _world(c, seed)
    Hxf, HS = _observed(w)
    d, out = w["yo"] - Hxf, []
    for i, k in ((0, w["surface"]), (w["surface"], w["m"])):
        n, x, r2 = k - i, d[i:k], w["rmse2"][i:k]
        if n == 0:
            out.append([0.0] + [math.nan] * 4)
            continue
        rd = x / r2
        out.append([float(n), float((x * x).mean().sqrt()), float(x.mean()),
                    float(((x * rd).sum() / n).sqrt()),
                    float(((HS[i:k].t() @ rd).square().sum() / n).sqrt())])
    return torch.tensor(out, dtype=torch.float64)


def _exact_operator(c, seed):
    """The weights of a cell split into simplices through the centres of its
    faces: along the order of |u - 1/2| the point lies between a corner, the
    centre of an edge, of a face and of the cell."""
    grids, var, pos, ax = _operator_inputs(c, seed)
    m, rows = len(var), []
    weights = {}
    for v, n in ((0, 3), (1, 2)):
        cell, u, ok = [], [], np.ones(m, bool)
        for k in range(n):
            i = np.clip(np.searchsorted(ax[k], pos[k], side="right") - 1, 0, len(ax[k]) - 2)
            cell.append(i)
            u.append((pos[k] - ax[k][i]) / (ax[k][i + 1] - ax[k][i]))
            ok &= (pos[k] >= ax[k][0]) & (pos[k] <= ax[k][-1])
        u = np.stack(u, 1)
        t = 2.0 * np.abs(u - 0.5)
        order = np.argsort(-t, axis=1, kind="stable")
        ts = np.concatenate([np.ones((m, 1)), np.take_along_axis(t, order, 1), np.zeros((m, 1))], 1)
        w = np.zeros((m, 2 ** n))
        state = grids[v]["state"]
        for j in range(2 ** n):
            bit = np.array([(j >> k) & 1 for k in range(n)])
            agree = np.take_along_axis((u >= 0.5) == (bit == 1), order, 1)
            for f in range(n + 1):  # the f largest coordinates fixed to the nearest side
                on = agree[:, :f].all(1)
                w[:, j] += np.where(on, (ts[:, f] - ts[:, f + 1]) / 2 ** (n - f), 0.0)
            ok &= state[tuple(cell[k] + bit[k] for k in range(n))] >= 0
        weights[v] = (w, ok)
    for l in range(m):
        w, ok = weights[int(var[l])]
        if ok[l]:
            rows.append(w[l])
    val = np.concatenate(rows) if rows else np.zeros(0)
    return [None, None, val, None]


def exact(case, seed):
    op = case["op"]
    if op == "operator":
        return _exact_operator(case, seed)
    if op == "fields":
        s = prepare(case, seed)
        state = s["files"][:, s["idx"]]
        out = s["out"]
        out[:, s["idx"]] = state
        return state, out
    if op == "nll":
        return _exact_nll(case, seed)
    if op == "report":
        return _exact_report(case, seed)
    return _exact_analysis(case, seed)

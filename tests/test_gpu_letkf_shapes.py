"""pb_letkf_analyse at the sizes where its kernel can go wrong, against the
LETKF oracle (oracle/letkf.py analyse_grid): 2, 16, 17 and 32 members (one
and two 16-member tiles, full and nearly empty), grids that leave rows and
columns of the last block unused, windows larger than the staging area in
rows and in columns, one attribute and more than sixteen, walls on both axes, on either
and on none, a negative variance (taken as any other number), accurate observations (a condition number of ~1e6), none at all, and NaN where
nothing is observed.

Tolerance: the analysis is x_mean + Wa X with |Wa| ~ 1; Wa's relative error is
eps times the condition number of Pa times a small factor (inverse square
root), 2.2e-16 * 1e6 * 16 = 4e-9 at the largest condition here, taken relative
to the increments; 1e-10 for the well-conditioned cases (1 + 605 / 0.01 / k)."""
import ctypes as C

import numpy as np
import pytest

from oracle import letkf as ol

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k,attrs,nx,ny,ox,oy,walls,var,tol", [
    (2, 1, 9, 7, 3, 5, (0, 0), 0.01, 1e-10), (16, 4, 17, 9, 5, 3, (0, 1), 0.01, 1e-10),
    (17, 2, 13, 6, 5, 5, (1, 1), 0.01, 1e-10), (32, 3, 19, 15, 13, 9, (0, 1), 0.01, 1e-10),
    (7, 2, 30, 33, 21, 31, (1, 1), 0.01, 1e-10), (3, 1, 300, 5, 291, 3, (0, 0), 0.01, 1e-10),
    (20, 1, 200, 4, 195, 1, (0, 1), 0.01, 1e-10), (5, 19, 12, 10, 3, 3, (0, 1), 0.01, 1e-10),
    (16, 2, 20, 11, 7, 7, (0, 1), 1e-6, 4e-9), (12, 1, 16, 16, 1, 1, (0, 0), 0.01, 1e-10),
    (16, 3, 18, 13, 5, 7, (1, 0), 0.01, 1e-10), (9, 2, 14, 11, 3, 3, (0, 0), -40.0, 1e-10)])
def test_letkf_shapes(k, attrs, nx, ny, ox, oy, walls, var, tol):
    import torch
    from pybella_amd import _abi
    print(f"case letkf shape k={k} attrs={attrs} {nx}x{ny} window {ox}x{oy}", flush=True)
    rng = np.random.default_rng(k * 1000 + nx)
    state = rng.standard_normal((k, attrs, nx, ny)) + 2.0
    obs = 2.0 + 0.5 * rng.standard_normal((attrs, nx, ny))
    mask = (rng.random((attrs, nx, ny)) < 0.3).astype(float)
    covar = var * rng.uniform(0.5, 2.0, attrs)
    loc = rng.random((ox, oy))
    bc = ol.boundary_mask((nx, ny), (not walls[0], not walls[1]), (ox - 1) // 2, (oy - 1) // 2)
    if walls == (1, 0):
        # beyond an x wall nothing is observed; the reference pads x with 0 and
        # then the periodic y with 1, which gives the corners back their weight
        px, py = (ox - 1) // 2, (oy - 1) // 2
        assert (bc[:px, :py] == 1).all() and (bc[:px, py:-py] == 0).all()
        bc[:px], bc[-px:] = 0.0, 0.0
    ref = ol.analyse_grid(state, obs, mask, covar, loc, bc, ox, oy, 1.05)
    ctx = _abi.default_context()
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    obs = np.where(mask != 0, np.nan, obs)       # never read where nothing is observed
    s, o, m = dev(state.swapaxes(2, 3)), dev(obs.swapaxes(1, 2)), dev(mask.swapaxes(1, 2))
    cv, lo, out = dev(covar), dev(loc), torch.full((k, attrs, ny, nx), np.nan, dtype=torch.float64, device="cuda")
    cfg = _abi.LetkfCfg(k, attrs, nx, ny, ox, oy, int(not walls[0]), int(not walls[1]), 1.05)
    call = lambda mm, res: ctx.check(ctx.lib.pb_letkf_analyse(
        ctx.h, C.byref(cfg), _abi.ptr(s), _abi.ptr(o), _abi.ptr(mm), _abi.ptr(cv), _abi.ptr(lo), _abi.ptr(res)), "letkf")
    call(m, out)
    got = out.cpu().numpy().swapaxes(2, 3)
    err = float(np.max(np.abs(got - ref)) / np.max(np.abs(ref)))
    assert err <= tol, err
    # nothing observed: the inflated ensemble
    call(torch.ones_like(m), out)
    free = state.mean(0) + np.sqrt(1.05) * (state - state.mean(0))
    err = float(np.max(np.abs(out.cpu().numpy().swapaxes(2, 3) - free)) / np.max(np.abs(free)))
    assert err <= 1e-13, err

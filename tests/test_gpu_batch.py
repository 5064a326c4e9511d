"""GPU tests of the batched uneven solves (pb_batch_*).

* FP64 (two-launch) batch: every member's solution and iteration count are
  bitwise those of the same member solved alone with the same tile height, on
  the chip (in one launch or several) and by launches per phase;
* mixed batch: every member reaches true relative residual 1e-8, and agrees
  with its single mixed solve to the tolerance;
* the batched projection step equals the single drop-in per member (<= 1e-7
  on the corrected momenta, as the drop-in's own parity bound);
* per member, the oracle's FP64 operator confirms the residual.
"""
import copy

import numpy as np
import pytest

from oracle import laplacian as olp
from pybella_amd import workloads as W

from _cases import oracle_op, rel

pytestmark = pytest.mark.gpu

SIZES = [(33, 17), (65, 33), (129, 65), (257, 129)]


def _members(per_size=2):
    out = []
    for nx, ny in SIZES:
        for m in range(per_size):
            out.append(W.batch_member_bubble(nx, ny, m))
    return out


def _systems(members):
    """(op, b) per member: operator assembled on the member's Sol0 and the
    scaled right-hand side of its projection, each on its own handle."""
    from pybella_amd import second_projection as sp
    ops, bs = [], []
    for Sol, Sol0, mpv, elem, node, ud, th in members:
        op = sp.Operator2D(sp.grid_of(node, ud))
        pr = sp._prepare(copy.deepcopy(Sol), copy.deepcopy(mpv), elem, node, ud, th, 0.05, copy.deepcopy(Sol0), op)
        ops.append(op)
        bs.append(pr.b)
    return ops, bs


@pytest.fixture(params=["resident", "launches"])
def route(request):
    """Both ways a batch runs; yields a check of the counts of a solve."""
    from pybella_amd import _abi
    ctx = _abi.default_context()
    ctx.set_resident(_abi.PB_RESIDENT_ON if request.param == "resident" else _abi.PB_RESIDENT_OFF)

    def check(solve):
        before = ctx.resident_runs()
        out = solve()
        n = {k: v - before[k] for k, v in ctx.resident_runs().items()}
        assert n["given_up"] == 0 and (n["declined"] if request.param == "resident" else n["runs"]) == 0, n
        assert n["runs"] + n["declined"] > 0
        return out

    yield check
    ctx.set_resident(_abi.PB_RESIDENT_ON)


def test_fp64_batch_equals_single_solves(route):
    import torch
    from pybella_amd.batch import BatchSolver
    print("case batch f64fast", flush=True)
    members = _members()
    ops, bs = _systems(members)
    for k, op in enumerate(ops):
        op.set_tile((2, 4, 8)[k % 3])          # uneven tiles across members
    singles = [op.solve(b, tol=1e-10, mode="f64fast") for op, b in zip(ops, bs)]
    singles = [(x.clone(), info) for x, info in singles]
    xs, infos = route(lambda: BatchSolver(ops).solve(bs, tol=1e-10, mode="f64fast"))
    torch.cuda.synchronize()
    for (xs1, i1), xb, ib in zip(singles, xs, infos):
        assert ib["info"] == 0 and ib["iters"] == i1["iters"], (ib, i1)
        assert torch.equal(xs1, xb)


def test_mixed_batch_converges_and_agrees(route):
    import torch
    from pybella_amd.batch import BatchSolver
    print("case batch mixed", flush=True)
    members = _members()
    ops, bs = _systems(members)
    xs, infos = route(lambda: BatchSolver(ops).solve(bs, tol=1e-8, mode="mixed"))
    for op, b, x, info in zip(ops, bs, xs, infos):
        assert info["info"] == 0 and info["true_rel_resid"] <= 1e-8, info
        xs1, i1 = op.solve(b, tol=1e-8, mode="mixed")
        # both are within 1e-8 of the exact solution in residual; compare modulo the null space
        d = (x - xs1).cpu().numpy()
        from oracle import nn as onn
        d = onn.project_null(d[None])[0]
        ref = onn.project_null(xs1.cpu().numpy()[None])[0]
        assert np.linalg.norm(d) <= 1e-5 * np.linalg.norm(ref)
    torch.cuda.synchronize()


def test_batched_projection_matches_single_dropin():
    from pybella_amd import second_projection as sp
    print("case batch impl_part", flush=True)
    members = _members(per_size=1)
    for m in members:
        m[5].tol = 1e-12      # both paths converge far below the comparison bound
    single = [copy.deepcopy(m) for m in members]
    batched = [copy.deepcopy(m) for m in members]
    for Sol, Sol0, mpv, elem, node, ud, th in single:
        sp.euler_backward_non_advective_impl_part(Sol, mpv, elem, node, ud, th, 0.0, 0.05, 1.0, Sol0=Sol0)
    infos = sp.euler_backward_non_advective_impl_part_batch(
        [(Sol, mpv, elem, node, ud, th, Sol0) for Sol, Sol0, mpv, elem, node, ud, th in batched], 0.05,
        mode="f64fast")
    assert all(i["info"] == 0 for i in infos)
    for a, b in zip(single, batched):
        for k in ("rhou", "rhov", "rhoX"):
            assert rel(getattr(b[0], k), getattr(a[0], k)) < 1e-7, k


def test_oracle_residual_per_member():
    print("case batch oracle residual", flush=True)
    from pybella_amd.batch import BatchSolver
    members = [W.batch_member_bubble(33, 17, 0), W.batch_member_bubble(65, 33, 1)]
    ops, bs = _systems(members)
    xs, infos = BatchSolver(ops).solve(bs, tol=1e-9, mode="mixed")
    for (Sol, Sol0, mpv, elem, node, ud, th), b, x, info in zip(members, bs, xs, infos):
        # the oracle operator on the same state the GPU assembled from (Sol0 after the ghost fill)
        from oracle import boundary as obd
        S0 = copy.deepcopy(Sol0)
        m2 = copy.deepcopy(mpv)
        obd.set_explicit_boundary_data(S0, elem, ud, th, m2)
        op_o, _, _ = oracle_op(S0, m2, elem, node, ud, th, 0.05)
        bb = b.cpu().numpy().ravel()
        r = bb - olp.lap2d(x.cpu().numpy().ravel(), op_o)
        assert np.linalg.norm(r) <= 2e-9 * np.linalg.norm(bb), (np.linalg.norm(r) / np.linalg.norm(bb), info)


@pytest.mark.parametrize("ry", [2, 5])
def test_flattened_batch_equals_single_solves(ry, route):
    """Uniform tile height: the batch runs one launch over every member's tiles,
    for the whole run or per phase; each member's iterates are still bitwise
    those of its own solve."""
    import torch
    from pybella_amd.batch import BatchSolver
    print(f"case flattened batch ry={ry}", flush=True)
    members = _members()
    ops, bs = _systems(members)
    for op in ops:
        op.set_tile(ry)
    singles = [op.solve(b, tol=1e-10, mode="f64fast") for op, b in zip(ops, bs)]
    singles = [(x.clone(), info) for x, info in singles]
    batch = BatchSolver(ops)
    for _ in range(2):   # by launches, the second solve replays the captured graph
        xs, infos = route(lambda: batch.solve(bs, tol=1e-10, mode="f64fast"))
        torch.cuda.synchronize()
        for (xs1, i1), xb, ib in zip(singles, xs, infos):
            assert ib["info"] == 0 and ib["iters"] == i1["iters"], (ib, i1)
            assert torch.equal(xs1, xb)
    xs, infos = route(lambda: batch.solve(bs, tol=1e-8, mode="mixed"))
    for op, b, info in zip(ops, bs, infos):
        assert info["info"] == 0 and info["true_rel_resid"] <= 1e-8, info


@pytest.mark.parametrize("mode", ["f64fast", "mixed"])
def test_mixed_heights_by_launches(mode):
    """Members of one size but several tile heights, by launches: kinds run in
    turn, each with a graph of its own; after a uniform batch of the same
    operators, and replayed over several solves."""
    import torch
    from pybella_amd import _abi
    from pybella_amd.batch import BatchSolver
    print(f"case batch mixed heights by launches {mode}", flush=True)
    ops, bs = _systems([W.batch_member_bubble(129, 65, m) for m in range(12)])
    ctx = ops[0].ctx
    try:
        for heights in ((4,), (2, 4, 8), (2, 3, 4, 5, 6, 8)):
            for k, op in enumerate(ops):
                op.set_tile(heights[k % len(heights)])
            ctx.set_resident(_abi.PB_RESIDENT_OFF)
            batch = BatchSolver(ops)
            for _ in range(3):
                xs, infos = batch.solve(bs, tol=1e-8, mode=mode)
            ctx.set_resident(_abi.PB_RESIDENT_ON)
            xr, ir = batch.solve(bs, tol=1e-8, mode=mode)
            for x, i, y, j in zip(xs, infos, xr, ir):
                assert i["info"] == 0 and i["iters"] == j["iters"] and torch.equal(x, y), (i, j)
    finally:
        ctx.set_resident(_abi.PB_RESIDENT_ON)


def test_batch_of_more_tiles_than_are_resident_at_once():
    """Twelve members of 85 tiles and four smaller ones, one group: their 1046
    tiles go in two launches, each member's result bitwise that of its own
    solve by launches per phase."""
    import torch
    from pybella_amd.batch import BatchSolver
    print("case batch in several launches", flush=True)
    members = [W.batch_member_bubble(257, 129, m) for m in range(12)]
    members[3:3] = [W.batch_member_bubble(nx, ny, 1) for nx, ny in SIZES[:2] * 2]
    ops, bs = _systems(members)
    for op in ops:
        op.set_tile(2)
    singles = [op.solve_noalloc(b, torch.full_like(b, np.nan), tol=1e-10, mode="f64fast") for op, b in zip(ops, bs)]
    batch, ctx = BatchSolver(ops), ops[0].ctx
    for _ in range(2):
        before = ctx.resident_runs()
        xs, infos = batch.solve(bs, tol=1e-10, mode="f64fast")
        n = {k: v - before[k] for k, v in ctx.resident_runs().items()}
        assert n == dict(runs=16, launches=2, declined=0, given_up=0), n
        for (x1, i1), x, i in zip(singles, xs, infos):
            assert i["info"] == 0 and i["iters"] == i1["iters"] and torch.equal(x1, x), (i, i1)

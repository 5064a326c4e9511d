"""The BiCGStab runs that stay on the chip (one launch per solve) against the
launch-per-phase iteration: same tiles, same operations, same summation
orders, so x, the iteration count and the info are bitwise equal.

``solve_noalloc`` always runs the launches, and the context's counts say that
``solve`` did not.  The grids cover a single tile,
tiles cut at the last row and column, wraps inside one tile, each way of
summing the records (one wave, several waves, class sums), more tiles than
two per compute unit, and a grid too large to be resident."""
import numpy as np
import pytest

from pybella_amd import workloads as W

pytestmark = pytest.mark.gpu


def _system(nx, ny, kind, seed=17):
    from pybella_amd import second_projection as sp
    Sol, mpv, elem, node, ud, th = W.stratified_state(nx, ny, compressible=kind != "psinc")
    if kind == "coriolis":
        ud.omega = 7.292e-5 * 50
        ud.derive()
    if kind == "xwall":
        ud.bdry_type[0] = W.BdryType.WALL
    op = sp.Operator2D(sp.grid_of(node, ud))
    rho, rhoY = sp.to_dev(Sol.rho), sp.to_dev(Sol.rhoY)
    op.assemble(sp.phys_of(ud, th), 0.05, rho, rhoY, rho, rhoY, sp.to_dev(sp.dSdy_cells(mpv, elem, node)))
    return op, op.scale_rhs(sp.to_dev(W.stratified_rhs(node, seed=seed)))


def _counted(op, solve):
    """solve(), and what it added to the context's counts of resident runs."""
    before = op.ctx.resident_runs()
    out = solve()
    return out, {k: n - before[k] for k, n in op.ctx.resident_runs().items()}


ONE = dict(runs=1, launches=1, declined=0, given_up=0)


def _same(op, b, **kw):
    import torch
    (x1, i1), n = _counted(op, lambda: op.solve(b, **kw))
    assert n == ONE, n
    x2, i2 = op.solve_noalloc(b, torch.full_like(b, np.nan), **kw)
    torch.cuda.synchronize()
    assert i1["iters"] == i2["iters"] and i1["info"] == i2["info"] and i1["half_step"] == i2["half_step"], (i1, i2)
    assert i1["resid"] == i2["resid"] and i1["bnrm2"] == i2["bnrm2"]
    assert torch.equal(x1, x2), float((x1 - x2).abs().max())
    return x1, i1


@pytest.mark.parametrize("mode", ["f64fast", "f64"])
@pytest.mark.parametrize("nx,ny,ry,kind", [
    (3, 3, 4, "psinc"), (9, 5, 2, "coriolis"), (64, 16, 4, "psinc"), (64, 32, 8, "coriolis"), (65, 17, 4, "psinc"),
    (66, 33, 4, "xwall"), (63, 31, 3, "coriolis"), (128, 64, 5, "comp"), (161, 81, 4, "psinc"), (300, 150, 2, "psinc"),
    (301, 151, 3, "xwall"), (513, 257, 4, "coriolis"), (513, 257, 2, "psinc"), (1025, 513, 6, "psinc")])
def test_resident_equals_launches(nx, ny, ry, kind, mode):
    print(f"case resident {kind} {nx}x{ny} ry {ry} {mode}", flush=True)
    op, b = _system(nx, ny, kind)
    op.set_tile(ry)
    for k in (1, 2, 9):   # short runs end at the iteration limit
        _same(op, b, tol=1e-30, maxiter=k, mode=mode)
    _, info = _same(op, b, tol=1e-8, maxiter=6000, mode=mode)
    assert info["info"] == 0 and info["true_rel_resid"] < 2e-8
    op.close()


@pytest.mark.parametrize("mode", ["f64fast", "f64"])
@pytest.mark.parametrize("nx,ny,tiles", [(509, 125, 64), (301, 205, 65), (509, 140, 72), (301, 301, 95),
                                         (509, 190, 96), (570, 170, 99)])
def test_class_sums_at_each_way_of_summing(nx, ny, tiles, mode):
    """Tile counts at the ends of each way of summing the records: one wave up
    to 64, two waves writing class sums of their own from 65 to 96, class sums
    formed by other blocks above."""
    print(f"case resident {tiles} tiles {mode}", flush=True)
    assert -(-nx // 64) * -(-ny // 16) == tiles
    op, b = _system(nx, ny, "coriolis")
    op.set_tile(4)
    for k in (1, 3, 60):
        _same(op, b, tol=1e-30, maxiter=k, mode=mode)
    op.close()


def test_more_tiles_than_two_per_unit_and_guess():
    """561 tiles of 16 rows (three blocks on some compute units), a given
    guess, a zero right-hand side and an exact one."""
    import torch
    print("case resident 1025x513 ry 4, guess, zero rhs", flush=True)
    op, b = _system(1025, 513, "coriolis")
    x, _ = _same(op, b, tol=1e-30, maxiter=40, mode="f64fast")
    (x1, i1), n = _counted(op, lambda: op.solve(b, tol=1e-8, maxiter=6000, mode="f64", x0=x))
    assert n == ONE, n
    x2, i2 = op.solve_noalloc(b, x.clone(), tol=1e-8, maxiter=6000, mode="f64", x0_given=True)
    assert i1["iters"] == i2["iters"] and torch.equal(x1, x2) and i1["info"] == 0
    z, iz = op.solve(torch.zeros_like(b), tol=1e-8, mode="f64fast")
    assert iz["info"] == 0 and iz["iters"] == 0 and float(z.abs().max()) == 0.0
    op.close()


def test_too_large_to_be_resident_and_two_streams():
    """1025 x 1025 with 2-row threads (8-row tiles, more than 768) runs by launches; solves
    from two threads, on their own contexts and streams and on the default
    one with an operator each, share the device's room."""
    import threading

    import torch
    from pybella_amd import _abi
    from pybella_amd import second_projection as sp
    print("case resident 1025x1025 ry 2, two threads", flush=True)
    op, b = _system(1025, 1025, "comp")
    op.set_tile(2)
    (x, info), n = _counted(op, lambda: op.solve(b, tol=1e-8, mode="f64fast"))
    assert n == dict(runs=0, launches=0, declined=1, given_up=0), n
    assert info["info"] == 0 and info["true_rel_resid"] < 2e-8
    op.close()
    op, b = _system(257, 129, "psinc")
    ref, _ = op.solve(b, mode="f64fast")
    torch.cuda.synchronize()
    got, err = [None] * 4, []

    def work(k):
        try:
            own = k < 2
            with torch.cuda.stream(torch.cuda.Stream() if own else torch.cuda.default_stream()):
                Sol, mpv, elem, node, ud, th = W.stratified_state(257, 129)
                o = sp.Operator2D(sp.grid_of(node, ud), ctx=_abi.Context(0) if own else None)
                rho, rhoY = sp.to_dev(Sol.rho), sp.to_dev(Sol.rhoY)
                dS = sp.to_dev(sp.dSdy_cells(mpv, elem, node))
                o.assemble(sp.phys_of(ud, th), 0.05, rho, rhoY, rho, rhoY, dS)
                for _ in range(5):
                    got[k], _ = o.solve(b, mode="f64fast")
                torch.cuda.synchronize()
                o.close()
        except Exception as e:   # noqa: BLE001
            err.append(e)

    for pair in ((0, 1), (2, 3)):
        ts = [threading.Thread(target=work, args=(k,)) for k in pair]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
    assert not err, err
    assert all(torch.equal(g, ref) for g in got)
    op.close()


@pytest.mark.parametrize("nx,ny,mode", [(61, 15, "f64"), (161, 81, "f64fast"), (161, 81, "mixed"), (301, 301, "f64"),
                                        (513, 257, "f64fast")])
def test_given_up_runs_are_repeated_by_launches(nx, ny, mode):
    """Every run given up by its abort word, set beforehand: blocks leave at
    their next wait (or end, x written), and the launches repeat the run.  Same
    solution as without, with and without a guess; the next solves go by
    launches at once, until the switch is set again."""
    import torch
    from pybella_amd import _abi
    print(f"case given up {nx}x{ny} {mode}", flush=True)
    op, b = _system(nx, ny, "coriolis")
    guess = torch.from_numpy(np.random.default_rng(3).standard_normal((ny, nx))).cuda()
    kws = [dict(tol=1e-8, mode=mode)] + ([dict(tol=1e-8, mode=mode, x0=guess)] if mode != "mixed" else [])
    ctx = op.ctx
    try:
        for kw in kws:
            ctx.set_resident(_abi.PB_RESIDENT_OFF)
            (x1, i1), n = _counted(op, lambda: op.solve(b, **kw))
            assert n["runs"] == n["given_up"] == 0 and n["declined"] >= 1, n
            ctx.set_resident(_abi.PB_RESIDENT_GIVE_UP)
            (x2, i2), n = _counted(op, lambda: op.solve(b, **kw))
            assert n["runs"] == 0 and n["given_up"] == 1, n
            assert i1["info"] == i2["info"] == 0 and i1["iters"] == i2["iters"] and torch.equal(x1, x2)
            (x2, i2), n = _counted(op, lambda: op.solve(b, **kw))
            assert n["runs"] == n["given_up"] == 0 and n["declined"] >= 1 and torch.equal(x1, x2), n
            ctx.set_resident(_abi.PB_RESIDENT_ON)
            (x2, i2), n = _counted(op, lambda: op.solve(b, **kw))
            assert n["runs"] >= 1 and n["declined"] == 0 and torch.equal(x1, x2), n
    finally:
        ctx.set_resident(_abi.PB_RESIDENT_ON)
    op.close()


def test_a_context_stops_trying_after_three_given_up_runs():
    """64 solves by launches after each given-up run, all after the third."""
    from pybella_amd import _abi
    print("case resident given up three times", flush=True)
    op, b = _system(33, 17, "psinc")
    ctx = op.ctx
    ref, _ = op.solve(b, mode="f64fast")
    try:
        ctx.set_resident(_abi.PB_RESIDENT_GIVE_UP)
        gave_up = []
        for k in range(3 * 65 + 70):
            _, n = _counted(op, lambda: op.solve(b, mode="f64fast"))
            assert n["runs"] == 0 and n["given_up"] + n["declined"] == 1
            gave_up += [k] * n["given_up"]
        assert gave_up == [0, 65, 130], gave_up
    finally:
        ctx.set_resident(_abi.PB_RESIDENT_ON)
    (x, _), n = _counted(op, lambda: op.solve(b, mode="f64fast"))
    assert n == ONE and bool((x == ref).all())
    op.close()


def test_a_grid_too_large_takes_no_memory_for_it():
    """2049 x 1025 nodes (2145 tiles) can never be resident: its solve, with a
    guess too, takes none of the exchange words (19 MB at this size)."""
    import torch
    print("case resident 2049x1025 memory", flush=True)
    op, b = _system(2049, 1025, "psinc")
    op.time_kernel(0, reps=1)   # the solver's vectors
    x, guess = torch.empty_like(b), torch.zeros_like(b)
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    for kw in (dict(mode="f64fast"), dict(mode="f64", x0=guess)):
        _, n = _counted(op, lambda: op.solve(b, x=x, tol=1e-30, maxiter=1, **kw))
        assert n["declined"] == 1 and n["runs"] == 0
    torch.cuda.synchronize()
    assert free - torch.cuda.mem_get_info()[0] < 12 << 20
    op.close()

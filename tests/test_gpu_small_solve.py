"""FP64 Jacobi-PCG of a small system in one launch: the same iterates, iterations and residuals bit for bit as
launch by launch (which a solve takes while the timer of its SpMV is on), and in find_pressure! and the
implicit viscous step."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _grid(lv, nx, ny, singular, periodic, jitter=0.1):
    dr = 1.0 / nx
    x = lv.inputs.jittered_lattice(nx, ny, dr, jitter=jitter, seed=0x5EED0A00 + nx)
    g = lv.VoronoiGrid(lv.Rectangle((0.0, 0.0), (1.0, ny * dr)), dr, xperiodic=periodic, yperiodic=periodic,
                       positions=x)
    lv.remesh(g)
    ic = lv.inputs.taylor_green(x, g.get("area"))
    for k in ("v", "rho", "mass", "P", "e", "mu"):
        g.set_soa(k, ic[k])
    if singular:
        g.set("c2", np.inf)
    else:
        lv.stiffened_eos(g, ic["gamma"], ic["P0"])
    return g, 0.1 * dr


def _by_launches(lv, grid, on):
    assert lv.lib().lv_timing_enable(grid.ctx, 1, int(on)) == 0


def _seen(lv, grid):
    c = ctypes.c_int64()
    assert lv.lib().lv_timing_seen(grid.ctx, 1, ctypes.byref(c)) == 0
    return c.value


# workgroups of 256 rows: one, partly empty, whole, one row more, and the most there are (256 of them);
# 0.45 dr of jitter gives rows of more than eight neighbours
@pytest.mark.parametrize("nx,ny,jitter", [(5, 3, 0.1), (16, 16, 0.1), (257, 1, 0.0), (24, 43, 0.45), (256, 256, 0.1)])
@pytest.mark.parametrize("singular,periodic", [(True, False), (False, True)])
def test_one_launch_equals_launch_by_launch(lv, gpu, nx, ny, jitter, singular, periodic):
    if periodic and min(nx, ny) < 8:
        periodic = False
    print("small solve %dx%d" % (nx, ny), flush=True)
    g, dt = _grid(lv, nx, ny, singular, periodic, jitter)
    s = lv.PressureSolver(g, method="pcg64", tol=1e-10, itmax=4000)
    s.assemble(dt)
    rng = np.random.default_rng(nx)
    b, x0 = rng.standard_normal(g.n), rng.standard_normal(g.n)
    nan = b.copy()
    nan[g.n // 2] = np.nan
    for rhs, guess, itmax in ((b, x0, 4000), (b, x0, 7), (np.zeros(g.n), np.zeros(g.n), 4000), (nan, x0, 50)):
        got = []
        for on in (1, 0):
            _by_launches(lv, g, on)
            x = s.solve(rhs, guess, raise_on_fail=False, itmax=itmax)
            got.append((x, s.last_stats, _seen(lv, g)))
        (xa, sa, na), (xb, sb, nb) = got
        assert na > 0 and nb == 0  # the timed solve ran launch by launch, the other did not
        assert np.array_equal(xa, xb, equal_nan=True)
        assert sa["iters"] == sb["iters"]
        for k in ("relres", "relres0"):
            assert np.array_equal(sa[k], sb[k], equal_nan=True)


def test_steps_equal_launch_by_launch(lv, gpu):
    """two steps! with ten Picard solves each, extrapolated guesses (which read the solve's residual) and the
    implicit viscous step on the same FP64 solver"""
    print("small solve in steps", flush=True)
    out = []
    for on in (1, 0):
        g, dt = _grid(lv, 40, 40, True, True)
        s = lv.PressureSolver(g, method="pcg64", tol=1e-10, itmax=4000, picard_window=4)
        d = lv.make_step_desc(dt, eos="rho", solver=s, viscous=lv.ViscousSolver(g, method="pcg64", tol=1e-9))
        _by_launches(lv, g, on)
        st = [lv.step_fused(g, d) for _ in range(2)]
        out.append((g.get_soa("x"), g.get_soa("P"), g.get_soa("v"), [k["iters"] for k in st]))
    assert all(np.array_equal(p, q) for p, q in zip(out[0][:3], out[1][:3])) and out[0][3] == out[1][3]


@pytest.mark.parametrize("tol", [1e-12, 1e-13])
@pytest.mark.parametrize("singular,periodic", [(True, False), (False, True)])
def test_the_true_residual_meets_the_tolerance(lv, gpu, tol, singular, periodic):
    """near what FP64 reaches the recurrence's residual falls below the tolerance before the true one does: the
    solve goes on from where it is until the true one has, on either route"""
    print("true residual %g" % tol, flush=True)
    g, dt = _grid(lv, 100, 100, singular, periodic)
    s = lv.PressureSolver(g, method="pcg64", tol=tol, itmax=20000)
    s.assemble(dt)
    for seed in range(6):
        b = np.random.default_rng(seed).standard_normal(g.n)
        got = []
        for on in (1, 0):
            _by_launches(lv, g, on)
            x = s.solve(b, np.zeros(g.n))
            assert s.last_stats["relres"][0] <= tol
            got.append((x, s.last_stats["iters"]))
        assert np.array_equal(got[0][0], got[1][0]) and got[0][1] == got[1][1]


def _looks(lv, grid, looks):
    """waits of at most so many looks from now on; how many solves gave up so far"""
    c = ctypes.c_int64()
    assert lv.lib().lv_test_small_solve(grid.ctx, looks, ctypes.byref(c)) == 0
    return c.value


# two workgroups, which often pass a sum that they wait a few looks for; and the most there are
@pytest.mark.parametrize("nx,ny,tries", [(32, 16, 400), (256, 256, 40)])
@pytest.mark.parametrize("singular", [True, False])
def test_a_solve_that_gives_up_starts_again_from_the_guess(lv, gpu, nx, ny, tries, singular):
    """whatever sum of it a workgroup gave up at, the last ones before and after the workgroups store their rows among them
    (one iteration, so that every sum has its turn): the launch-by-launch solve of the guess, its mean too, bit for bit"""
    print("small solve gives up %dx%d" % (nx, ny), flush=True)
    g, dt = _grid(lv, nx, ny, singular, False)
    s = lv.PressureSolver(g, method="pcg64", tol=1e-10)
    s.assemble(dt)
    rng = np.random.default_rng(nx)
    b, x0 = rng.standard_normal(g.n), rng.standard_normal(g.n)
    for itmax in (1, 2):
        _by_launches(lv, g, 1)
        want = s.solve(b, x0, raise_on_fail=False, itmax=itmax)
        _by_launches(lv, g, 0)
        before = _looks(lv, g, 0)
        for k in range(tries):
            _looks(lv, g, k // 10)
            x = s.solve(b, x0, raise_on_fail=False, itmax=itmax)
            assert np.array_equal(x, want), "looks %d" % (k // 10)
            assert s.last_stats["iters"][0] == itmax
        gave_up = _looks(lv, g, -1) - before
        print("small solve gave up %d of %d" % (gave_up, tries), flush=True)
        assert gave_up > 0
    if singular:
        assert abs(want.mean() - x0.mean()) < 1e-12


def test_solves_after_one_that_gave_up_do_not_wait_again(lv, gpu):
    print("small solve rests", flush=True)
    g, dt = _grid(lv, 100, 100, True, False)
    s = lv.PressureSolver(g, method="pcg64", tol=1e-10, itmax=4000)
    s.assemble(dt)
    b = np.random.default_rng(3).standard_normal(g.n)
    want = s.solve(b, np.zeros(g.n))
    before = _looks(lv, g, 0)
    for _ in range(30):
        assert np.array_equal(s.solve(b, np.zeros(g.n)), want)
    assert _looks(lv, g, -1) == before + 1

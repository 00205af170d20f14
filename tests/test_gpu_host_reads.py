"""What the host reads of the device while it launches on: the couplings' count against their room, the error of a
move behind the remesh it leads to, the items of a list that outgrew its buffer."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _lattice(lv, K, jitter, seed=0x5EED0F00):
    return lv.inputs.jittered_lattice(K, K, 1.0 / K, jitter=jitter, seed=seed)


def _operator(lv, grid, dt):
    solver = lv.PressureSolver(grid, method="amg", tol=1e-8)
    solver.assemble(dt)
    return solver.operator()


@pytest.mark.parametrize("K", [24, 90])
def test_more_couplings_than_the_room_of_the_first_operator(lv, oracle, gpu, K):
    """a regular lattice's four a row, then a jittered one's six, in the same grid: the operator of a fresh grid"""
    print("couplings %d" % K, flush=True)
    out = []
    for first in (True, False):
        grid = lv.VoronoiGrid(lv.UnitRectangle(), 1.0 / K, xperiodic=True, yperiodic=True,
                              positions=_lattice(lv, K, 0.0 if first else 0.4))
        for x in ([_lattice(lv, K, 0.0), _lattice(lv, K, 0.4)] if first else [_lattice(lv, K, 0.4)]):
            grid.set_positions(x)
            lv.remesh(grid)
            n = grid.n
            for name, v in (("rho", 1.0), ("mass", 1.0 / n), ("c2", 2500.0), ("mu", 1e-3)):
                grid.set(name, np.full(n, v))
            op = _operator(lv, grid, 1e-3)
        out.append(op)
    for a, b in zip(*out):
        assert np.array_equal(a, b)
    assert out[0][1][-1] > 5 * grid.n


@pytest.mark.parametrize("bad", ["one", "all"])
def test_a_move_with_nan_velocity_is_refused_and_the_grid_lives_on(lv, gpu, bad):
    print("nan move %s" % bad, flush=True)
    K = 20
    x = _lattice(lv, K, 0.2)
    grid = lv.VoronoiGrid(lv.UnitRectangle(), 1.0 / K, xperiodic=True, yperiodic=True, positions=x)
    lv.remesh(grid)
    want = grid.mesh()
    v = np.zeros(2 * grid.n)
    v[7 if bad == "one" else slice(None)] = np.nan
    grid.set("v", v)
    with pytest.raises(lv.LVError, match="Velocity field invalidated"):
        lv.move(grid, 1e-3)
    with pytest.raises(lv.LVError):
        grid.mesh()
    grid.set_positions(x)
    lv.remesh(grid)
    for a, b in zip(grid.mesh(), want):
        assert np.array_equal(a, b)
    fresh = lv.VoronoiGrid(lv.UnitRectangle(), 1.0 / K, xperiodic=True, yperiodic=True, positions=x)
    lv.remesh(fresh)
    for g in (grid, fresh):
        g.set("v", np.full(2 * g.n, 0.25))
        lv.move(g, 1e-3)
    for a, b in zip(grid.mesh(), fresh.mesh()):
        assert np.array_equal(a, b)


def test_more_seeds_than_the_first_list(lv, gpu):
    """a small set, then a large one in the same grid: the first list of the large set does not fit"""
    print("larger set", flush=True)
    xs = [_lattice(lv, K, 0.3) for K in (30, 100)]
    grid = lv.VoronoiGrid(lv.UnitRectangle(), 1.0 / 30, r_max=0.5, capacity=10000, positions=xs[0])
    for x in xs:
        grid.set_positions(x)
        lv.remesh(grid)
    fresh = lv.VoronoiGrid(lv.UnitRectangle(), 1.0 / 30, r_max=0.5, positions=xs[1])
    lv.remesh(fresh)
    for a, b in zip(grid.mesh(), fresh.mesh()):
        assert np.array_equal(a, b)
    for a, b in zip(grid.cell_list(), fresh.cell_list()):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("K", [20, 190, 320])
def test_a_refused_move_leaves_the_polygons_of_the_last_remesh(lv, gpu, tmp_path, K):
    print("refused move %d" % K, flush=True)
    grid = lv.VoronoiGrid(lv.UnitRectangle(), 1.0 / K, xperiodic=True, yperiodic=True, positions=_lattice(lv, K, 0.45))
    lv.remesh(grid)
    area = grid.get("area")
    polygons = open(lv.export_grid(grid, str(tmp_path / "before")), "rb").read()
    v = np.full(2 * grid.n, 0.25)
    v[5] = np.nan
    grid.set("v", v)
    with pytest.raises(lv.LVError, match="Velocity field invalidated"):
        lv.move(grid, 0.5 / K)
    assert np.array_equal(grid.get("area"), area)
    assert open(lv.export_grid(grid, str(tmp_path / "after")), "rb").read() == polygons

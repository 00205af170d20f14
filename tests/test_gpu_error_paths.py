"""Calls that end in the middle (no memory: lv_test_fail makes a point fail as an allocation does) leave nothing behind:
the next call gives what a context gives that never failed."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CELL_LIST_ROOM, CELL_LIST, ASSEMBLY, AMG_COUNTS, AMG_LEVELS, OPERATOR_ROOM, WHOLE_STAGE, STAGE = range(1, 9)


def _fail(lv, grid, point):
    assert lv.lib().lv_test_fail(grid.ctx, point) == 0


def _grid(lv, K=48, c2=2500.0, remesh=True):
    x = lv.inputs.jittered_lattice(K, K, 1.0 / K, jitter=0.2, seed=0x5EED1100)
    grid = lv.VoronoiGrid(lv.UnitRectangle(), 1.0 / K, positions=x)
    if remesh:
        lv.remesh(grid)
        _set(lv, grid, c2)
    return grid


def _set(lv, grid, c2):
    for name, v in (("rho", 1.0), ("mass", 1.0 / grid.n), ("c2", c2), ("mu", 1e-3)):
        grid.set(name, np.full(grid.n, v))


def _same(a, b):
    return len(a) == len(b) and all(np.array_equal(p, q) for p, q in zip(a, b))


def test_a_refused_move_without_room_for_its_list(lv, gpu):
    """the move's error is not the next remesh's"""
    print("fails: room of the list behind a refused move", flush=True)
    grid = _grid(lv, remesh=False)
    v = np.zeros(2 * grid.n)
    v[3] = np.nan
    grid.set("v", v)
    _fail(lv, grid, CELL_LIST_ROOM)
    with pytest.raises(lv.LVError):
        lv.move(grid, 1e-3)
    lv.remesh(grid)
    assert _same(grid.mesh(), _grid(lv).mesh())


@pytest.mark.parametrize("point", [CELL_LIST_ROOM, CELL_LIST])
def test_a_remesh_that_ends_in_the_middle(lv, gpu, point):
    print("fails: remesh at %d" % point, flush=True)
    grid = _grid(lv, remesh=False)
    for again in range(2):  # (the second time there is a list already)
        if point == CELL_LIST or again == 0:
            _fail(lv, grid, point)
            with pytest.raises(lv.LVError):
                lv.remesh(grid)
            with pytest.raises(lv.LVError):
                grid.mesh()
        lv.remesh(grid)
        fresh = _grid(lv)
        assert _same(grid.mesh(), fresh.mesh()) and _same(grid.cell_list(), fresh.cell_list())


def test_an_assembly_that_ends_in_the_middle(lv, gpu):
    """a compressible one, then an incompressible system: singular, its solution with the guess's mean"""
    print("fails: assembly", flush=True)
    out = []
    for failed in (True, False):
        grid = _grid(lv)
        s = lv.PressureSolver(grid, method="pcg64", tol=1e-10, itmax=2000)
        if failed:
            _fail(lv, grid, ASSEMBLY)
            with pytest.raises(lv.LVError):
                s.assemble(1e-3)
        grid.set("c2", np.inf)
        s.assemble(1e-3)
        b = np.random.default_rng(1).standard_normal(grid.n)
        out.append((s.solve(b, np.full(grid.n, 0.5)),) + tuple(s.operator()))
    assert _same(*out)
    assert abs(out[0][0].mean() - 0.5) < 1e-12


@pytest.mark.parametrize("point", [AMG_COUNTS, AMG_LEVELS])
@pytest.mark.parametrize("c2", [2500.0, np.inf])
def test_a_multilevel_set_up_that_ends_in_the_middle(lv, gpu, point, c2):
    print("fails: multilevel set-up at %d" % point, flush=True)
    out = []
    for failed in (True, False):
        grid = _grid(lv, c2=c2)
        s = lv.PressureSolver(grid, method="amg", tol=1e-8)
        s.assemble(1e-3)
        b = np.random.default_rng(2).standard_normal(grid.n)
        for again in range(2):  # (the second time the work space is there)
            if failed:
                _fail(lv, grid, point)
                with pytest.raises(lv.LVError):
                    s.solve(b, np.zeros(grid.n))
            x = s.solve(b, np.zeros(grid.n))
            lv.remesh(grid)
            s.assemble(1e-3)
        out.append((x, np.array(s.last_stats["iters"])))
    assert _same(*out)


def test_an_operator_without_room(lv, gpu):
    """the couplings' old room is gone and there is no new: no operator, until an assembly finds room (one of as many
    couplings as the old room held, which is no longer there)"""
    print("fails: room of the operator", flush=True)
    K = 48
    few = lv.inputs.jittered_lattice(K, K, 1.0 / K, jitter=0.0, seed=1)  # four couplings a row
    grid = _grid(lv, K)
    s = lv.PressureSolver(grid, method="amg", tol=1e-8)
    b = np.random.default_rng(3).standard_normal(grid.n)
    grid.set_positions(few)
    lv.remesh(grid)
    _set(lv, grid, 2500.0)
    s.assemble(1e-3)
    many = lv.inputs.jittered_lattice(K, K, 1.0 / K, jitter=0.4, seed=2)
    grid.set_positions(many)
    lv.remesh(grid)
    _set(lv, grid, 2500.0)
    _fail(lv, grid, OPERATOR_ROOM)
    with pytest.raises(lv.LVError):
        s.assemble(1e-3)
    with pytest.raises(lv.LVError, match="not assembled"):
        s.solve(b, np.zeros(grid.n))
    with pytest.raises(lv.LVError, match="not assembled"):
        s.operator()
    for x in (few, many):
        out = []
        for g in (grid, _grid(lv, K)):
            g.set_positions(x)
            lv.remesh(g)
            _set(lv, g, 2500.0)
            t = lv.PressureSolver(g, method="amg", tol=1e-8)
            t.assemble(1e-3)
            out.append((t.solve(b, np.zeros(g.n)),) + tuple(t.operator()))
        assert _same(*out)


@pytest.mark.parametrize("point", [WHOLE_STAGE, STAGE])
def test_read_outs_without_room_for_their_staging(lv, gpu, tmp_path, point):
    """in smaller pieces, or through the context's own work space; a call's scratch in memory of its own"""
    print("fails: staging %d" % point, flush=True)
    K = 300
    q = np.random.default_rng(4).random((5000, 2))

    def grid_of():
        grid = _grid(lv, K)
        grid.set_soa("D", np.random.default_rng(5).standard_normal(4 * grid.n))
        grid.set_soa("v", np.random.default_rng(6).standard_normal(2 * grid.n))
        return grid

    reads = [lambda g: g.mesh(), lambda g: (g.get("v"), g.get("D")), lambda g: (lv.point_value(g, q, "v[1]"),),
             lambda g: (lv.nearest_polygon(g, q),), lambda g: (lv.movingls(lv.QuadraticExpansion, g, "v[2]"),),
             lambda g: (np.frombuffer(open(lv.export_grid(g, str(tmp_path / "f"), "v"), "rb").read(), np.uint8),)]
    whole = grid_of()
    for k, read in enumerate(reads):
        grid = grid_of()
        _fail(lv, grid, point)
        assert _same(read(grid), read(whole)), k

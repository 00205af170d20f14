"""The ways clipping runs (a group of lanes per seed up to 32768 seeds and for polygons that outgrow a thread's
slots; a thread per seed above, with ten slots up to 98304 seeds and eight beyond): mesh bit for bit the oracle's on
either side of the lines, on regular, strongly jittered and random seeds."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _same_mesh(lv, oracle, x, dr, periodic, r_max=None):
    grid = lv.VoronoiGrid(lv.UnitRectangle(), dr, r_max=r_max, xperiodic=periodic, yperiodic=periodic, positions=x)
    lv.remesh(grid)
    op = oracle.Particles(oracle.Grid((0.0, 0.0), (1.0, 1.0), dr, r_max=r_max, xperiodic=periodic,
                                      yperiodic=periodic), x)
    op.remesh()
    for a, b in zip(grid.mesh(), op.mesh()):
        assert np.array_equal(a, b)
    assert np.array_equal(grid.get("area"), op.area())
    return grid


@pytest.mark.parametrize("periodic", [True, False])
@pytest.mark.parametrize("K,jitter", [(12, 0.1), (17, 0.45), (40, 0.0), (221, 0.45), (222, 0.45)])
def test_mesh_of_lattices_bit_exact(lv, oracle, gpu, K, jitter, periodic):
    print("clip lattice %d %g" % (K, jitter), flush=True)
    x = lv.inputs.jittered_lattice(K, K, 1.0 / K, jitter=jitter, seed=0x5EED0B00 + K)
    grid = _same_mesh(lv, oracle, x, 1.0 / K, periodic)
    assert (grid.n <= 49152) == (K < 222)
    if jitter > 0.4:  # some polygons need more than eight slots
        assert np.max(np.diff(grid.mesh()[0])) > 8


@pytest.mark.parametrize("n", [1, 2, 900, 49152, 49153])
def test_mesh_of_random_seeds_bit_exact(lv, oracle, gpu, n):
    print("clip random %d" % n, flush=True)
    x = np.random.default_rng(n).random(2 * n)
    _same_mesh(lv, oracle, x, 0.2 if n < 900 else 1.0 / np.sqrt(n), False, r_max=3.0 if n < 900 else None)


@pytest.mark.parametrize("around,ok", [(12, True), (40, False)])
def test_polygons_of_too_many_edges_raise(lv, oracle, gpu, around, ok):
    """a seed inside a ring of seeds: as many edges, at most LV_MAX_EDGES = 16"""
    print("clip ring %d" % around, flush=True)
    t = 2 * np.pi * (np.arange(around) + 0.1) / around
    ring = 0.5 + 0.2 * np.stack([np.cos(t), np.sin(t)])
    x = np.concatenate([[0.5], ring[0], [0.5], ring[1]])
    if ok:
        _same_mesh(lv, oracle, x, 0.1, False, r_max=2.0)
    else:
        grid = lv.VoronoiGrid(lv.UnitRectangle(), 0.1, r_max=2.0, positions=x)
        with pytest.raises(lv.LVError, match="LV_MAX_EDGES"):
            lv.remesh(grid)


@pytest.mark.parametrize("n,seed", [(50001, 1), (65536, 2), (57344 + 255, 3)])
def test_mesh_of_uneven_chunks_bit_exact(lv, oracle, gpu, n, seed):
    """a thread per seed, the last chunk of 256 seeds and the last group of chunks not full; half of the cells empty"""
    print("clip chunks %d" % n, flush=True)
    x = np.random.default_rng(seed).random(2 * n)
    _same_mesh(lv, oracle, x, 0.5 / np.sqrt(n), True, r_max=9.0 / np.sqrt(n))


@pytest.mark.parametrize("periodic", [True, False])
@pytest.mark.parametrize("K", [181, 182, 313, 314])
def test_mesh_at_the_lines_between_the_ways(lv, oracle, gpu, K, periodic):
    print("clip line %d" % K, flush=True)
    x = lv.inputs.jittered_lattice(K, K, 1.0 / K, jitter=0.45, seed=0x5EED0B80 + K)
    grid = _same_mesh(lv, oracle, x, 1.0 / K, periodic)
    assert (grid.n <= 32768) == (K == 181) and (grid.n <= 98304) == (K < 314)


def _clip_ms(lv, n, h):
    import ctypes

    grid = lv.VoronoiGrid(lv.UnitRectangle(), 1.0 / np.sqrt(n), h=h, r_max=3.0,
                          positions=np.random.default_rng(n).random(2 * n))
    lv.remesh(grid)
    assert lv.lib().lv_timing_enable(grid.ctx, 2, 1) == 0
    lv.remesh(grid)
    ms, count = ctypes.c_double(), ctypes.c_int64()
    assert lv.lib().lv_timing_read(grid.ctx, 2, ctypes.byref(ms), ctypes.byref(count), None) == 0
    assert count.value == 1
    return ms.value


def test_crowded_cells_are_read_once_by_a_group(lv, oracle, gpu):
    """Every seed in one cell, 2,000 and then 8,000 of them.  Four times the candidates for a seed, and its groups' 2,000
    wavefronts share the 1,024 SIMDs, two to each, where 500 had one to themselves: at most eight times as long, if a
    group lists each candidate once.  (Reading the cell anew for every 64 of its candidates makes it 16 times the
    reads a seed.)"""
    print("clip crowded", flush=True)
    few, many = (min(_clip_ms(lv, n, 1.0) for _ in range(3)) for n in (2000, 8000))
    print("clip crowded: %.2f ms, %.2f ms" % (few, many), flush=True)
    assert many <= 8.0 * few
    x = np.random.default_rng(5).random(2 * 3000)
    grid = lv.VoronoiGrid(lv.UnitRectangle(), 1.0 / np.sqrt(3000), h=0.5, r_max=3.0, positions=x)
    lv.remesh(grid)
    op = oracle.Particles(oracle.Grid((0.0, 0.0), (1.0, 1.0), 1.0 / np.sqrt(3000), h=0.5, r_max=3.0), x)
    op.remesh()
    for a, b in zip(grid.mesh(), op.mesh()):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("n,h,periodic", [(32768, 2.0, False), (32769, 2.0, False), (98304, 2.0, False), (98305, 2.0, False),
                                          (98304 + 255, 1.0, True), (131073, 1.0, True)])
def test_mesh_of_random_seeds_at_the_lines_between_the_ways(lv, oracle, gpu, n, h, periodic):
    """random seeds, whose polygons outgrow a thread's slots far more often than a lattice's: on either side of both lines,
    and with eight slots a last chunk and a last group of chunks that are not full"""
    print("clip random line %d" % n, flush=True)
    x = np.random.default_rng(n).random(2 * n)
    dr = h / 2.0 / np.sqrt(n)  # cells of h / sqrt(n)
    _same_mesh(lv, oracle, x, dr, periodic, r_max=9.0 / np.sqrt(n))

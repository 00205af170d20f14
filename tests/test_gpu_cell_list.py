"""The cell list where its counting sort can go wrong: cells on both sides of the one-workgroup scan, cells of many
labels, several images of a seed in one cell, and more images than the first buffer holds."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _same(lv, oracle, x, dr, xmax=(1.0, 1.0), periodic=(False, False), **kw):
    grid = lv.VoronoiGrid(lv.Rectangle((0.0, 0.0), xmax), dr, xperiodic=periodic[0], yperiodic=periodic[1],
                          positions=x, **kw)
    op = oracle.Particles(oracle.Grid((0.0, 0.0), xmax, dr, xperiodic=periodic[0], yperiodic=periodic[1], **kw), x)
    for _ in range(2):  # the second list starts from what the first left of the counters
        lv.remesh(grid)
        start, labels = grid.cell_list()
        want_start, want_labels = op.grid.cell_list(x)
        assert np.array_equal(start, want_start)
        assert np.array_equal(labels, want_labels)
    return start, labels


@pytest.mark.parametrize("periodic", [(False, False), (True, True)])
@pytest.mark.parametrize("K,small", [(3, True), (33, True), (228, True), (260, False)])
def test_cells_on_both_sides_of_the_scan_line(lv, oracle, gpu, K, small, periodic):
    print("cell list %d" % K, flush=True)
    x = lv.inputs.jittered_lattice(K, K, 1.0 / K, jitter=0.4, seed=0x5EED0C00 + K)
    start, _ = _same(lv, oracle, x, 1.0 / K, periodic=periodic)
    assert (start.size <= 16384) == small


@pytest.mark.parametrize("K,h", [(10, 0.5), (10, 2.5)])
@pytest.mark.parametrize("periodic", [(False, False), (True, False), (True, True)])
def test_crowded_cells(lv, oracle, gpu, K, h, periodic):
    print("crowded cells %d %g" % (K, h), flush=True)
    x = lv.inputs.jittered_lattice(K, K, 1.0 / K, jitter=0.3, seed=0x5EED0D00 + K)
    start, labels = _same(lv, oracle, x, 1.0 / K, periodic=periodic, h=h)
    assert np.max(np.diff(start)) >= (16 if h < 1.0 else 100)
    if h > 1.0 and periodic[0]:
        assert np.any(np.diff(labels) == 0)


def test_more_images_than_the_first_buffer(lv, oracle, gpu):
    """a strip as wide as r_max: every seed has two images beside it"""
    print("cell list strip", flush=True)
    dr = 1.0 / 2000
    x = lv.inputs.jittered_lattice(10, 2000, dr, jitter=0.3, seed=0x5EED0E00)
    n = x.size // 2
    _, labels = _same(lv, oracle, x, dr, xmax=(10 * dr, 1.0), periodic=(True, False))
    assert labels.size > n + n // 4 + 4096


def test_no_seed_in_the_grid_is_refused(lv, gpu):
    print("cell list empty", flush=True)
    grid = lv.VoronoiGrid(lv.UnitRectangle(), 0.1, positions=np.full(20, 1e3))
    with pytest.raises(lv.LVError, match="no items"):
        lv.remesh(grid)

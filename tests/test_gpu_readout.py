"""Read-outs of every size: by the runtime's copy, by the staged one (3 MiB and more, several pieces and threads), and
of more rows than the staging holds."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _grid(lv, n, seed=0):
    rng = np.random.default_rng(seed)
    grid = lv.VoronoiGrid(lv.UnitRectangle(), 0.01, positions=rng.random(2 * n))
    planes = {k: rng.standard_normal(c * n) for k, c in (("P", 1), ("v", 2), ("D", 4))}
    for k, a in planes.items():
        grid.set_soa(k, a)
    return grid, planes


@pytest.mark.parametrize("n", [1, 7, 4096, 98304, 98305, 262144, 600011, 1300003])
def test_fields_by_planes_and_by_rows(lv, gpu, n):
    print("read-out %d" % n, flush=True)
    grid, planes = _grid(lv, n)
    for k, a in planes.items():
        assert np.array_equal(grid.get_soa(k), a)
    assert np.array_equal(grid.get("P"), planes["P"])
    assert np.array_equal(grid.get("v"), planes["v"].reshape(2, n).T)
    D = grid.get("D")
    assert D.shape == (n, 2, 2) and D.flags["C_CONTIGUOUS"]
    assert np.array_equal(D, planes["D"].reshape(2, 2, n).transpose(2, 1, 0))  # column-major planes


def test_read_outs_of_several_grids_at_once(lv, gpu):
    """a thread for each of four contexts"""
    print("read-outs at once", flush=True)
    grids = [_grid(lv, 300000 + 1000 * k, seed=k) for k in range(4)]
    wrong = []

    def work(k):
        grid, planes = grids[k]
        for _ in range(5):
            for name, a in planes.items():
                if not np.array_equal(grid.get_soa(name), a):
                    wrong.append((k, name))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong

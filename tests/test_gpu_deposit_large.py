"""Grids of 4096 tiles and more, with wide footprints: few (added to the grid
cell by cell), many (tile by tile, several runs of 64 groups of 64 particles)
and a mixture with narrow ones, against the oracle; a footprint across the whole
grid among them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _torch():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


def _close(g, go, what):
    # offsets of up to 4100 cells carry 4100 float64 roundings on each axis, and a
    # weight's slope is at most 3 per h >= 1 cell: 6e-12 of the largest value,
    # whose sums are of one sign
    err = np.abs(g - go).max() / np.abs(go).max()
    print(what, "max error over the largest cell", err, flush=True)
    assert err <= 1e-11


# wide particles, their cells a side, narrow particles
MAPS = [(0, 0, 500), (1, 34, 0), (300, 100, 0), (40, 150, 300), (65, 400, 0), (6000, 42, 100)]
VOLS = [(0, 0, 300), (1, 10, 0), (40, 30, 200), (60, 95, 0), (6000, 21, 100)]


@pytest.mark.parametrize("wide,cells,narrow", MAPS)
@pytest.mark.parametrize("cons", [False, True])
def test_map_of_many_tiles(oracle, wide, cells, narrow, cons):
    torch = _torch()
    from meshoid_amd import engine

    print("large map", wide, cells, narrow, cons, flush=True)
    res, size = 4100, 10.0
    rng = np.random.default_rng(wide + cells)
    n = wide + narrow
    dx = size / (res - 1)
    pos = rng.random((n, 3)) * size
    h = np.where(np.arange(n) < wide, 0.5 * cells * dx, 2 * dx) * (1 + 0.02 * rng.standard_normal(n))
    if wide == 40:
        h[0] = 0.6 * size
    order = rng.permutation(n)
    pos, h, f = pos[order], np.maximum(h[order], 2 * size / res), rng.random(n) + 0.1
    td = lambda a: torch.from_numpy(a).cuda()
    g = engine.surface_density(td(f), td(pos), td(h), np.array([5.0] * 3), size, res, 1.0, cons)
    go = oracle.grid_surface_density(f, pos, h, np.array([5.0] * 3), size, res, conservative=cons)
    _close(g.cpu().numpy(), go, "map")


@pytest.mark.parametrize("wide,cells,narrow", VOLS)
@pytest.mark.parametrize("periodic", [False, True])
def test_volume_of_many_tiles(oracle, wide, cells, narrow, periodic):
    torch = _torch()
    from meshoid_amd import engine

    print("large volume", wide, cells, narrow, periodic, flush=True)
    res, size = 260, 10.0
    rng = np.random.default_rng(wide + cells)
    n = wide + narrow
    dx = size / (res - 1)
    pos = rng.random((n, 3)) * size
    h = np.where(np.arange(n) < wide, 0.5 * cells * dx, 1.2 * dx) * (1 + 0.02 * rng.standard_normal(n))
    if wide == 40:
        h[0] = 0.55 * size
    order = rng.permutation(n)
    pos, h, f = pos[order], np.maximum(h[order], dx), rng.random(n) + 0.1
    td = lambda a: torch.from_numpy(a).cuda()
    g = engine.grid_density(td(f), td(pos), td(h), np.array([5.0] * 3), size, res, periodic, dx)
    go = oracle.grid_density(f, pos, h, np.array([5.0] * 3), size, res, size if periodic else -1.0)
    _close(g.cpu().numpy(), go, "volume")

"""Neighbourhood windows that begin in a bitmap tile without occupied cells and hold a cell of the next tile:
grids whose rows lie across the ends of the popcount scan's tiles (2048 words), in a level of two nodes, after a
build that has left other prefixes in the same memory."""
import numpy as np
import pytest

import oracle_binding as O
from octree_amd import api
from octree_amd import workloads as W
from parity import compare, fetch, gpu_build, synthetic, weighted_color_check

pytestmark = pytest.mark.gpu

TILE_BITS = 32 * 2048
PER_CELL = 6


def _cell_coords(cell, g):
    """Coordinates of a cell index: 4 x 4 pencils of x-rows."""
    row, x = divmod(cell, g)
    pencil, inside = divmod(row, 16)
    p = (g + 3) // 4
    return x, (pencil % p) * 4 + inside % 4, (pencil // p) * 4 + inside // 4


def _sparse_cloud(g, seed):
    """float64 records in the unit cube: of the two opposite octants' grids, cells at the first bits of every
    second tile (the tiles before them are empty) and the cells next to them in the row."""
    per_node = g ** 3  # g is a multiple of 4
    rng = np.random.default_rng(seed)
    xyz = []
    for at in range(TILE_BITS, 2 * per_node, 2 * TILE_BITS):
        node, cell = divmod(at + int(rng.integers(0, 2)), per_node)
        for c in (cell, cell + 1):
            assert c < per_node
            corner = np.array(_cell_coords(c, g), np.float64) + 0.2 + 0.6 * rng.random((PER_CELL, 3))
            xyz.append((corner / g + node) * 0.5)
    xyz = np.concatenate(xyz)
    n = len(xyz)
    out = np.empty((n, 27), np.uint8)
    out[:, :24] = np.ascontiguousarray(xyz).view(np.uint8).reshape(n, 24)
    out[:, 24:] = rng.integers(0, 256, (n, 3))
    return out.reshape(-1), n


@pytest.mark.parametrize("weighted", [False, True], ids=["inter", "weighted"])
@pytest.mark.parametrize("g", [96, 100])
def test_window_across_an_empty_tile(g, weighted):
    cloud, n = _sparse_cloud(g, seed=g)
    build = W.BuildSpec(4, 20, 8.0, g, inter=True, weighted=weighted)
    cubic, scale = [0.0, 0.0, 0.0, 1.0, 1.0, 1.0], [1e-6] * 3
    before, spec, before_box = synthetic(200_000, 1, seed=g)
    orc = O.build(cloud, n, 27, 1, cubic, scale, build, keep=weighted)
    assert np.count_nonzero(orc.internal) == 3, "two nodes and the root subsample"
    print(f"case prefix windows g {g} weighted {weighted} n {n}", flush=True)
    s = api.Session(0)
    try:
        gpu_build(before, spec.points, spec.stride, 1, before_box, [spec.scale] * 3, build, sess=s)
        gpu_build(cloud, n, 27, 1, cubic, scale, build, sess=s)
        got = fetch(s)
        compare(got, orc, check_colors=not weighted)
        if weighted:
            # one thread sums a cell's few weights: no order to differ by, but the weights are floats here and
            # doubles in the oracle, so an average next to a whole number may fall to its other side
            weighted_color_check(got, orc.handle, tol=1)
    finally:
        s.close()
        if orc.handle is not None:
            orc.handle.close()

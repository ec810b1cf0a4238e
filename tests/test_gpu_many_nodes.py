"""Levels of very many internal nodes: more tiles and leaf chunks than one launch takes (and more children than
a launch of eight per node could have work-items for), and a level in more node batches than are read back at
a time."""
import numpy as np
import pytest

import oracle_binding as O
from octree_amd import workloads as W
from parity import check_against_oracle, fetch, gpu_build

pytestmark = pytest.mark.gpu


def _cloud(xyz, seed):
    """float64 records of the given points with random colours."""
    n = len(xyz)
    out = np.empty((n, 27), np.uint8)
    out[:, :24] = np.ascontiguousarray(xyz, np.float64).view(np.uint8).reshape(n, 24)
    out[:, 24:] = np.random.default_rng(seed).integers(0, 256, (n, 3))
    return out.reshape(-1)


@pytest.mark.parametrize("weighted", [False, True], ids=["inter", "weighted"])
def test_more_nodes_than_a_launch_takes(weighted):
    n, grid = (3 << 20) + 5, 512
    xyz = np.random.default_rng(7).random((n, 3)) * [1.0, 1.0, 0.25]
    cloud, cubic, scale = _cloud(xyz, 8), [0.0, 0.0, 0.0, 1.0, 1.0, 1.0], [1e-6] * 3
    build = W.BuildSpec(grid, 1, 4.0, 2, inter=True, weighted=weighted)
    orc = O.build(cloud, n, 27, 1, cubic, scale, build, threads=8, keep=weighted)
    level0, level1 = np.count_nonzero(orc.key < grid ** 3), np.count_nonzero(orc.key < grid ** 3 + (grid // 2) ** 3)
    assert level0 > 1 << 21, "one launch takes all tiles"
    assert (level1 - level0) * 8 * 256 > 1 << 32, "a tile per child slot fits a launch"
    print(f"case many nodes weighted {weighted} level 0 {level0} level 1 {level1 - level0}", flush=True)
    s = gpu_build(cloud, n, 27, 1, cubic, scale, build)
    try:
        check_against_oracle(fetch(s), orc, weighted)
    finally:
        s.close()
        if orc.handle is not None:
            orc.handle.close()


def test_level_in_more_batches_than_are_read_back():
    """A node's bitmap and prefix take 256 MiB at g = 1024, so a batch holds 24 nodes and 64 batches 1536. The
    expected subsamples are computed here (the oracle would hold g^3 cells a node): coordinates are multiples of
    2^-20 in a cube of 64, so cells are exact, and the point with the smallest index wins a cell."""
    grid, g, threshold, n = 64, 1024, 12, 120_000
    rng = np.random.default_rng(3)
    xy = rng.random((n, 2)) * 64
    z = 20 + 12 * np.sin(xy[:, 0] / 9) * np.cos(xy[:, 1] / 7) + rng.random(n)
    xyz = np.floor(np.column_stack([xy, z]) * 2.0 ** 20) / 2.0 ** 20
    alive, want = np.ones(n, bool), []
    for level in range(1, 7):
        side = 2.0 ** level  # of a node at this level, in the coordinates' unit
        at = (xyz // side).astype(np.int64)
        node = at @ [1, grid >> level, (grid >> level) ** 2]
        inner = np.bincount(node, minlength=(grid >> level) ** 3) >= threshold
        cell = np.floor((xyz - at * side) * (g / side)).astype(np.int64) @ [1, g, g * g]
        inputs = np.nonzero(alive & inner[node])[0]
        order = np.lexsort((inputs, cell[inputs], node[inputs]))
        inputs = inputs[order]
        first = np.ones(len(inputs), bool)
        first[1:] = (np.diff(node[inputs]) != 0) | (np.diff(cell[inputs]) != 0)
        kept = inputs[first]
        alive &= ~inner[node]
        alive[kept] = True
        if level == 1:
            assert np.count_nonzero(inner) > 24 * 64, "the level's batches are read back at once"
        want.append(np.sort(node[kept] * n + kept))
    print(f"case many batches n {n}", flush=True)
    s = gpu_build(_cloud(xyz, 4), n, 27, 1, [0.0, 0.0, 0.0, 64.0, 64.0, 64.0], [2.0 ** -20] * 3,
                  W.BuildSpec(grid, threshold, 12.0, g))
    try:
        _, nodes, lut, _ = fetch(s)
        offset = np.cumsum([0] + [(grid >> l) ** 3 for l in range(7)])
        for level in range(1, 7):
            ids = np.nonzero(nodes.internal & (nodes.key >= offset[level]) & (nodes.key < offset[level + 1]))[0]
            got = [(int(nodes.key[i]) - int(offset[level])) * n +
                   lut[int(nodes.data_idx[i]):int(nodes.data_idx[i]) + int(nodes.point_count[i])].astype(np.int64) for i in ids]
            np.testing.assert_array_equal(np.sort(np.concatenate(got)), want[level - 1], f"level {level}")
    finally:
        s.close()

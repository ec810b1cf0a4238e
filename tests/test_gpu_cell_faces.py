"""Points on and beside the faces of grid cells: the builds take a point's cell from a product unless the
product lies close to a whole number, and from the division it stands for then."""
import numpy as np
import pytest

from octree_amd import workloads as W
from parity import run_case, synthetic

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cloud_type", [0, 1])
@pytest.mark.parametrize("grid,sub,offset", [(64, 16, 0.0), (32, 12, -733.1)])
def test_points_at_cell_faces(cloud_type, grid, sub, offset):
    n = 30_011
    cloud, spec, cubic = synthetic(n, cloud_type, seed=grid + cloud_type, offset=offset)
    dtype, width = (np.float32, 12) if cloud_type == 0 else (np.float64, 24)
    records = cloud.reshape(n, spec.stride)
    xyz = np.ascontiguousarray(records[:, :width]).view(dtype)
    lo, hi = xyz.min(0).copy(), xyz.max(0).copy()
    rng = np.random.default_rng(grid)
    # faces of the dense grid and of the node grids of the first levels, then up to two neighbours of them,
    # then distances around the one from which the product decides
    cell = (cubic[3] - cubic[0]) / (grid * sub)
    on = np.asarray(cubic[:3]) + np.round((xyz.astype(np.float64) - np.asarray(cubic[:3])) / cell) * cell
    on += cell * np.exp2(rng.integers(-34, -26, (n, 1))) * rng.integers(-1, 2, (n, 1)) * (rng.random((n, 1)) < 0.5)
    face = on.astype(dtype)
    for step in range(2):
        move = rng.integers(0, 3, (n, 3))
        face = np.where(move == 1, np.nextafter(face, dtype(np.inf)), np.where(move == 2, np.nextafter(face, dtype(-np.inf)), face))
    inside = np.clip(face, lo, hi)
    records[:, :width] = inside.astype(dtype).view(np.uint8).reshape(n, width)
    print(f"case cell faces type {cloud_type} grid {grid} sub {sub}", flush=True)
    run_case(np.ascontiguousarray(records).reshape(-1), n, spec.stride, cloud_type, cubic, [spec.scale] * 3,
             W.BuildSpec(grid, 400, 3.0, sub, intra=True))

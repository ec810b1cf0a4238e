"""Subsampling grids whose cells of a leaf take fewer bits of a Morton code than a bitmap word has: leaves of more
points than one workgroup orders, and of a few."""
import pytest

from octree_amd import workloads as W
from parity import run_case, synthetic

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("g", [4, 8, 16, 32, 64])
@pytest.mark.parametrize("n,grid,threshold,mode", [(120_000, 2, 20_000, {}), (60_000, 64, 300, {"intra": True, "random": True})],
                         ids=["full-leaves", "small-leaves"])
def test_small_subsampling_grids(g, n, grid, threshold, mode):
    cloud, spec, cubic = synthetic(n, 1, box=(20.0, 20.0, 20.0), seed=g)
    print(f"case small grids g {g} G {grid}", flush=True)
    run_case(cloud, n, spec.stride, 1, cubic, [spec.scale] * 3, W.BuildSpec(grid, threshold, 6.0, g, **mode), threads=8)

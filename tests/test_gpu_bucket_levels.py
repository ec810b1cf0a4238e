"""Grids on both sides of the one from which the sort's buckets are finer, in clouds whose buckets are
sparse, crowded (more points than one workgroup sorts) and a single one."""
import pytest

from octree_amd import workloads as W
from parity import run_case, synthetic

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid", [64, 128, 256, 512])
@pytest.mark.parametrize("n,box,clusters", [(40_000, (30.0, 30.0, 30.0), 0), (700_000, (2000.0, 2000.0, 2000.0), 1)],
                         ids=["sparse", "crowded"])
def test_bucket_levels(grid, n, box, clusters):
    cloud, spec, cubic = synthetic(n, 0, box=box, clusters=clusters, seed=grid)
    print(f"case bucket levels grid {grid} n {n}", flush=True)
    run_case(cloud, n, spec.stride, 0, cubic, [spec.scale] * 3, W.BuildSpec(grid, 3000, 3.5, 32, inter=True), threads=8)

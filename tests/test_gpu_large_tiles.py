"""Builds from the size on whose levels combine tiles of inputs in LDS, where a tile's table can go wrong:
every input in a cell of its own, nearly all inputs in a few cells, grids whose words straddle rows."""
import pytest

from octree_amd import workloads as W
from parity import run_case, synthetic

pytestmark = pytest.mark.gpu

LARGE_POINTS = 3 << 20


@pytest.mark.parametrize("n,cloud_type,box,clusters,build", [
    (LARGE_POINTS - 1, 0, (50.0, 50.0, 50.0), 0, W.BuildSpec(128, 20_000, 3.0, 128, intra=True)),
    (LARGE_POINTS, 0, (50.0, 50.0, 50.0), 0, W.BuildSpec(128, 20_000, 3.0, 128, intra=True)),
    (LARGE_POINTS, 1, (4000.0, 4000.0, 10.0), 2, W.BuildSpec(64, 3000, 3.0, 20, inter=True, random=True, seed=3)),
    (LARGE_POINTS + 777, 0, (4000.0, 4000.0, 10.0), 1, W.BuildSpec(128, 5000, 3.0, 6)),
], ids=["below", "spread", "crowded-inter", "crowded-small-grid"])
def test_tiles_combined_in_lds(n, cloud_type, box, clusters, build):
    cloud, spec, cubic = synthetic(n, cloud_type, box=box, clusters=clusters, seed=5)
    print(f"case large tiles {n} type {cloud_type} box {box} clusters {clusters} g {build.subsampling_grid}", flush=True)
    run_case(cloud, n, spec.stride, cloud_type, cubic, [spec.scale] * 3, build, threads=8)

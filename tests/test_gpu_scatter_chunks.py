"""The bucket scatter's chunk sizes: clouds around the sizes where the points per thread change, and around
whole chunks of the large ones."""
import pytest

from octree_amd import workloads as W
from parity import run_case, synthetic

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cloud_type", [0, 1])
@pytest.mark.parametrize("n", [1025, (1 << 17), (1 << 17) + 1, (1 << 19), (1 << 19) + 1, 86 * 6144, 86 * 6144 + 1])
def test_scatter_chunks(n, cloud_type):
    cloud, spec, cubic = synthetic(n, cloud_type, seed=n % 97)
    print(f"case scatter chunks {n} type {cloud_type}", flush=True)
    run_case(cloud, n, spec.stride, cloud_type, cubic, [spec.scale] * 3, W.BuildSpec(128, 2000, 3.0, 32, intra=True),
             threads=8)

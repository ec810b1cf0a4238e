"""A build whose subsampled points do not fit the output fails at the level that finds it, with the levels
below built and the ones above without work; the same session then builds the cloud."""
import dataclasses

import pytest

import oracle_binding as O
from octree_amd import api
from octree_amd import workloads as W
from parity import compare, fetch, gpu_build, synthetic

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [30_000, 3 << 20], ids=["small", "large"])
@pytest.mark.parametrize("factor", [1.0, 1.3])
def test_rebuild_after_a_level_that_does_not_fit(n, factor):
    cloud, spec, cubic = synthetic(n, 0, box=(50.0, 50.0, 20.0), seed=23)
    build = W.BuildSpec(128, max(200, n // 500), 4.0, 32 if n < 1 << 20 else 128, intra=True)
    orc = O.build(cloud, n, spec.stride, 0, cubic, [spec.scale] * 3, build, threads=8)
    assert orc.used > factor * n, "the case does not overflow"
    print(f"case overflow {n} factor {factor}", flush=True)
    s = api.Session(0)
    try:
        with pytest.raises(api.OctreeError):
            gpu_build(cloud, n, spec.stride, 0, cubic, [spec.scale] * 3, dataclasses.replace(build, output_factor=factor), sess=s)
        gpu_build(cloud, n, spec.stride, 0, cubic, [spec.scale] * 3, build, sess=s)
        compare(fetch(s), orc)
    finally:
        s.close()

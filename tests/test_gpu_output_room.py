"""Builds with next to no room for subsampled points: what a service charges for one, and the arrays that hold no
more cells than the output has room for."""
import dataclasses

import pytest

import oracle_binding as O
from octree_amd import api
from octree_amd import workloads as W
from parity import check_against_oracle, compare, fetch, gpu_build, synthetic

pytestmark = pytest.mark.gpu


def _charged(n, grid, g, threshold):
    """Bytes that a build of n 15-byte records from host memory is charged whose output holds n records."""
    dense = sum((grid >> l) ** 3 for l in range(grid.bit_length()))
    nodes = min(dense, grid.bit_length() * n)
    return (15 * n + 8 * dense + 4 * ((dense + 31) // 32)  # cloud; counts and ids, occupancy bits
            + 85 * nodes + n // 1024 + 22 * n  # nodes, leaf chunks; point indices and records
            + (2 * 20 + 2 + 4) * n + (2 * n // 196608 + 1) * (8 + 4 * 32768)  # sorted records, split buckets
            + 34 + 8 + 32 * n + 32  # a staged point; inputs of a level, a cell
            + 8 * (g ** 3 // 32) * min(nodes, n // threshold + 8))  # bitmaps and prefixes


def test_service_takes_a_build_that_stages_nothing():
    """The root is the only leaf, so an output of n records is enough; a budget of what the build is charged
    without room for subsampled points takes it."""
    n, grid, g, threshold = 3_000_001, 64, 32, 1 << 22
    cloud, spec, cubic = synthetic(n, 0, seed=5)
    build = W.BuildSpec(grid, threshold, 1.0, g, intra=True)
    orc = O.build(cloud, n, spec.stride, 0, cubic, [spec.scale] * 3, build, threads=8)
    assert orc.used == n
    print("case service with an output of n records", flush=True)
    with api.Service(slots=1, memory_budget=_charged(n, grid, g, threshold)) as service:
        s = api.Session(0)
        try:
            s.set_cloud(cloud, n, spec.stride, 0, cubic, [spec.scale] * 3)
            s.configure(build)
            service.submit(s)
            service.wait(s)
            compare(fetch(s), orc)
        finally:
            s.close()


@pytest.mark.parametrize("mode", [{}, {"inter": True}, {"inter": True, "weighted": True}], ids=["none", "inter", "weighted"])
@pytest.mark.parametrize("n", [30_000, 3 << 20], ids=["small", "large"])
def test_levels_with_more_cells_than_the_output_has_room_for(n, mode):
    cloud, spec, cubic = synthetic(n, 0, box=(50.0, 50.0, 20.0), seed=29)
    build = W.BuildSpec(128, max(200, n // 500), 4.0, 32 if n < 1 << 20 else 128, **mode)
    orc = O.build(cloud, n, spec.stride, 0, cubic, [spec.scale] * 3, build, threads=8, keep=bool(mode.get("weighted")))
    s = api.Session(0)
    try:
        for factor in (1.0, 1.0 + 4.0 / n, 1.2):
            assert orc.used > factor * n, "the case does not overflow"
            print(f"case output room {n} {mode} factor {factor}", flush=True)
            with pytest.raises(api.OctreeError, match="output"):
                gpu_build(cloud, n, spec.stride, 0, cubic, [spec.scale] * 3,
                          dataclasses.replace(build, output_factor=factor), sess=s)
        gpu_build(cloud, n, spec.stride, 0, cubic, [spec.scale] * 3, build, sess=s)
        check_against_oracle(fetch(s), orc, bool(mode.get("weighted")), sample_nodes=60)
    finally:
        s.close()
        if orc.handle is not None:
            orc.handle.close()

"""The distance-weighted filter around cells that hold a good part of the cloud (coincident points): the lanes
that are left walk one long run of points together."""
import numpy as np
import pytest

from octree_amd import workloads as W
from parity import run_case, synthetic

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cloud_type,random", [(0, False), (1, True)])
@pytest.mark.parametrize("crowd", [1, 3, 4, 5, 67, 6000])
def test_coincident_points(cloud_type, random, crowd):
    """Colours within one of the oracle's: both add up to 6000 weights of at most 1 in 32 bits, an error of
    at most 6000 * 2^-24 of the sums, 0.1 of a channel."""
    n = 12_000
    cloud, spec, cubic = synthetic(n, cloud_type, seed=crowd)
    width = 12 if cloud_type == 0 else 24
    records = cloud.reshape(n, spec.stride)
    at = np.random.default_rng(crowd).permutation(n)[:crowd]
    lo = records[:, :width].copy().view(np.float32 if cloud_type == 0 else np.float64)
    keep = np.setdiff1d(np.arange(n), np.concatenate([lo.argmin(0), lo.argmax(0)]))  # the box stays
    at = keep[np.isin(keep, at)]
    records[at, :width] = records[keep[0], :width]
    print(f"case coincident points {len(at)} type {cloud_type}", flush=True)
    run_case(np.ascontiguousarray(records).reshape(-1), n, spec.stride, cloud_type, cubic, [spec.scale] * 3,
             W.BuildSpec(32, 500, 4.0, 16, inter=True, weighted=True, random=random, seed=3))

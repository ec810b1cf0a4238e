"""Records as the kernels read them from a cloud: strides from the smallest to past the staged ones,
clouds that start anywhere in a 16-byte word, sizes around a workgroup's records."""
import ctypes

import numpy as np
import pytest

from hip_memory import DeviceBuffer
from octree_amd import api
from octree_amd import workloads as W
from parity import run_case, synthetic

pytestmark = pytest.mark.gpu


def _restrided(cloud, stride, wide, offset=0):
    """The records of `cloud` with `wide` bytes each, `offset` bytes into the buffer, noise in between."""
    n = len(cloud) // stride
    rng = np.random.default_rng(wide)
    out = rng.integers(0, 256, offset + n * wide, dtype=np.uint8)
    keep = min(stride, wide)
    out[offset:].reshape(n, wide)[:, :keep] = cloud.reshape(n, stride)[:, :keep]
    return out


@pytest.mark.parametrize("fn", ["ocpi_compute_bounding_box", "ocpi_compute_bounding_box_noalloc"])
@pytest.mark.parametrize("cloud_type,strides", [(0, (12, 15, 16, 31, 32, 33, 40)), (1, (24, 27, 29, 32, 33, 48))])
def test_bounding_box_of_any_stride_and_start(fn, cloud_type, strides):
    call = getattr(api.library(), fn)
    width = 12 if cloud_type == 0 else 24
    for n in (1, 511, 512, 513, 1700):
        cloud, spec, _ = synthetic(n, cloud_type, seed=n, offset=-300.0)
        xyz = cloud.reshape(n, spec.stride)[:, :width].copy().view("<f4" if cloud_type == 0 else "<f8").astype(np.float64)
        want = np.concatenate([xyz.min(0), xyz.max(0)])
        for stride in strides:
            for offset in (0, 1, 6, 15):
                buf = DeviceBuffer(_restrided(cloud, spec.stride, stride, offset))
                real, cubic = np.zeros(6), np.zeros(6)
                try:
                    rc = call(buf.ptr.value + offset, n, stride, cloud_type, 0, real.ctypes.data, cubic.ctypes.data)
                finally:
                    buf.close()
                assert rc == 0, api.last_error()
                np.testing.assert_array_equal(real, want, f"n {n} stride {stride} offset {offset}")


@pytest.mark.parametrize("cloud_type,stride", [(0, 16), (0, 32), (0, 37), (1, 29), (1, 32), (1, 41)])
def test_build_of_any_stride(cloud_type, stride):
    cloud, spec, cubic = synthetic(20_011, cloud_type)
    print(f"case stride {stride}", flush=True)
    run_case(_restrided(cloud, spec.stride, stride), spec.points, stride, cloud_type, cubic, [spec.scale] * 3,
             W.BuildSpec(64, 500, 3.0, 16, intra=True))

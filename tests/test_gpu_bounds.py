"""The bounding box's two passes: sizes around its workgroups and around the most of them, and calls from several
threads at once, each on a cloud of its own."""
import threading

import numpy as np
import pytest

from hip_memory import DeviceBuffer
from octree_amd import api

pytestmark = pytest.mark.gpu

FUNCTIONS = ["ocpi_compute_bounding_box", "ocpi_compute_bounding_box_noalloc"]


def _box(fn, buf, n):
    real, cubic = np.zeros(6), np.zeros(6)
    rc = getattr(api.library(), fn)(buf.ptr.value, n, 15, 0, 0, real.ctypes.data, cubic.ctypes.data)
    assert rc == 0, api.last_error()
    return real


def _cloud(n, seed):
    xyz = np.random.default_rng(seed).normal(size=(n, 3)).astype(np.float32)
    records = np.zeros((n, 15), np.uint8)
    records[:, :12] = xyz.view(np.uint8).reshape(n, 12)
    return DeviceBuffer(records.reshape(-1)), np.concatenate([xyz.min(0), xyz.max(0)]).astype(np.float64)


@pytest.mark.parametrize("fn", FUNCTIONS)
@pytest.mark.parametrize("n", [1, 255, 256, 257, 256 * 1024 - 1, 256 * 1024, 256 * 1024 + 1, 3_000_001])
def test_sizes_around_the_workgroups(fn, n):
    buf, want = _cloud(n, n)
    try:
        for _ in range(3):
            np.testing.assert_array_equal(_box(fn, buf, n), want)
    finally:
        buf.close()


@pytest.mark.parametrize("fn", FUNCTIONS)
def test_calls_from_several_threads(fn):
    clouds = [_cloud(1000 + 40_000 * k, k) for k in range(7)]
    wrong = []

    def work(k):
        for _ in range(50):
            got = _box(fn, clouds[k][0], 1000 + 40_000 * k)
            if not np.array_equal(got, clouds[k][1]):
                wrong.append((k, got))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(len(clouds))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for buf, _ in clouds:
        buf.close()
    assert not wrong, wrong[:3]

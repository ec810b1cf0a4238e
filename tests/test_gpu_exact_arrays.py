"""Builds from the size on whose level arrays are sized level by level from what the host reads back: equal to the
oracle, for the filters that keep other arrays, and in the memory that the levels need."""
import ctypes
import os
import time

import numpy as np
import pytest

import oracle_binding as O
from octree_amd import workloads as W
from hip_memory import hip
from parity import check_against_oracle, fetch, gpu_build

pytestmark = [pytest.mark.gpu, pytest.mark.timeout(900)]

POINTS = (1 << 27) + 3
THREADS = min(os.cpu_count() or 1, 16)


@pytest.fixture(scope="module")
def cloud():
    spec = W.CloudSpec(POINTS, 0, (600.0, 600.0, 90.0), 24, 41)
    data = W.generate(spec)
    return data, spec, W.bounding_box(data, POINTS, spec.stride, 0)[1]


def _free():
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def _level_most(orc, grid):
    """The most inputs and the most occupied cells of a level."""
    starts = np.cumsum([0] + [(grid >> l) ** 3 for l in range(grid.bit_length())])
    level = np.searchsorted(starts, orc.key, side="right") - 1
    most = [0, 0]
    for l in range(1, grid.bit_length()):
        nodes = np.nonzero(orc.internal & (level == l))[0]
        children = orc.children[nodes].reshape(-1)
        most = np.maximum(most, [orc.point_count[children[children >= 0]].sum(), orc.point_count[nodes].sum()])
    return int(most[0]), int(most[1])


@pytest.mark.parametrize("mode", [{"intra": True, "random": True}, {"inter": True, "weighted": True}], ids=["intra", "weighted"])
def test_level_arrays_as_read_back(cloud, mode):
    data, spec, cubic = cloud
    t0 = time.time()
    build = W.BuildSpec(128, 20_000, 2.0, 64, **mode)
    weighted = "weighted" in mode
    orc = O.build(data, POINTS, spec.stride, 0, cubic, [spec.scale] * 3, build, threads=THREADS, keep=weighted)
    print(f"  [{time.time() - t0:6.1f} s] oracle built: {len(orc.key):,} nodes, {orc.used:,} records", flush=True)
    print(f"case exact arrays {mode}", flush=True)
    before = _free()
    s = gpu_build(data, POINTS, spec.stride, 0, cubic, [spec.scale] * 3, build)
    try:
        # cloud, sorted records twice, codes and permutation; output; staging; inputs and cells of the largest
        # level; and what does not grow with the points or does so slowly (bitmaps, split buckets, dense grid)
        records = s.summary()["capacity"]
        inputs, cells = _level_most(orc, 128)
        need = POINTS * (15 + 2 * 20 + 6) + 22 * records + 34 * (records - POINTS) + \
            (32 * inputs + 16 * cells if weighted else 4 * inputs + 24 * cells)
        assert before - _free() < need + (1 << 30), (before - _free(), need)
        check_against_oracle(fetch(s), orc, weighted, sample_nodes=60)
        print(f"  [{time.time() - t0:6.1f} s] compared", flush=True)
    finally:
        s.close()
        if orc.handle is not None:
            orc.handle.close()

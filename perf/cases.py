"""The work that users of the octree builder have it do, as cases that can be timed and compared.

Four kinds of call:
  build     a whole octree of one cloud that lies in HBM: ocpi_generate_octree on an initialised
            session. The octree stays in HBM until a program exports or copies it.
  host      one cloud from host memory to its octree in host memory: upload (ocpi_init_octree),
            build, copies of the nodes, the point LUT and the output records.
  batch     many small clouds built together by the batched pipeline (ocpi_batch_build), which
            leaves every octree in host memory.
  bounds    the bounding box of a cloud in HBM (ocpi_compute_bounding_box), a caller's step before
            its first build of a cloud.

Clouds are a heightfield plus Gaussian clusters in random order (terrestrial and aerial scans), the
shape of the package's own synthetic workloads, made on the GPU from the seed.

The order of the points inside one octree node is free (a node holds a set of points), so the
fields of a result come with every node's records in ascending order of their point index. Records
are followed by zeros up to the output's capacity, as in an exported octree.bin, and nodes by zeros
up to the most that a cloud of this size can have, so that a case's fields always have one shape.
The distance-weighted filter's colours are averages of real weights, whose last unit depends on the
order of the additions; they come as (16-bit) numbers, all other fields as whole numbers.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "octree-cuda_amd"))

from octree_amd import api  # noqa: E402
from octree_amd.workloads import BuildSpec  # noqa: E402

STRIDE = {"f32": 15, "f64": 27}
CLOUD_TYPE = {"f32": 0, "f64": 1}
# the reference's command line passes the scale as a float
SCALE = {"f32": float(np.float32(0.001)), "f64": float(np.float32(0.01))}
FILTERS = ("none", "intra", "inter", "weighted")
# records an octree holds per input point (subsampled points included): 2.0 to 2.45 on these clouds
RECORDS_PER_POINT = 2.3


def _cloud(points, dtype, side, height, clusters, sigma, offset):
    return {"points": points, "dtype": dtype, "side": side, "height": height, "clusters": clusters, "sigma": sigma,
            "offset": offset}


def _build(name, cloud, chunking, subsampling, threshold, color, explicit, kind="build", factor=3.0):
    return {"name": name, "kind": kind, **cloud, "chunking_grid": chunking, "subsampling_grid": subsampling,
            "threshold": threshold, "filter": color, "explicit": explicit, "output_factor": factor}


def listed():
    coin = _cloud(5_138_448, "f32", 100.0, 20.0, 8, 2.0, 0.0)
    heidentor = _cloud(25_836_417, "f32", 50.0, 30.0, 16, 2.0, 0.0)
    morrowbay = _cloud(119_701_547, "f64", 2000.0, 150.0, 64, 2.0, 1e6)
    served = (400.0, 60.0, 24, 2.0)  # the serving loop's clouds
    return [
        # a preview of a small object: the smallest build, bound by launches and size readbacks
        _build("preview 50K f32 first", _cloud(50_003, "f32", 20.0, 4.0, 4, 0.5, 0.0), 64, 32, 2000, "none", False),
        # the small request of a tile server, at the default grids: the 512^3 pyramid outweighs the points
        _build("request 200K f64 intra", _cloud(200_017, "f64", *served, 1e6), 512, 128, 10000, "intra", False),
        # a middling request at the batched builds' grids, explicit winners, no filter
        _build("request 1.5M f64 explicit", _cloud(1_500_007, "f64", 300.0, 60.0, 8, 3.0, 1e5), 256, 64, 5000,
               "none", True),
        # one scanned object (the reference's coin): implicit, inter-cell average
        _build("coin 5.1M f32 inter", coin, 512, 128, 10000, "inter", False),
        # the largest request a server takes: explicit, distance-weighted filter
        _build("request 20M f64 weighted", _cloud(20_000_000, "f64", *served, 1e6), 512, 128, 10000, "weighted", True),
        # a scanned building (the reference's heidentor): explicit, intra-cell average
        _build("heidentor 25.8M f32 intra", heidentor, 512, 128, 10000, "intra", True),
        # an aerial scan (the reference's morrowbay), the headline build: implicit, weighted
        _build("morrowbay 119.7M f64 weighted", morrowbay, 512, 128, 10000, "weighted", False),
        # the coin from a file's bytes to the octree that an exporter writes out
        _build("coin host to host", coin, 512, 128, 10000, "inter", False, kind="host"),
        # a tile job: many small clouds of either type at once, in HBM
        {"name": "batch of 64, 10K to 400K", "kind": "batch", "clouds": 64, "least": 10_000, "most": 400_000,
         "chunking_grid": 256, "subsampling_grid": 64, "threshold": 5000, "filter": "inter", "explicit": False,
         "output_factor": 3.0},
        # the bounding box before a small and before a large build
        {"name": "bounds 200K f32", "kind": "bounds", **_cloud(200_017, "f32", *served, 0.0)},
        {"name": "bounds 119.7M f64", "kind": "bounds", **morrowbay},
    ]


def _log(rng, least, most):
    return int(math.exp(rng.uniform(math.log(least), math.log(most))))


def draw(rng):
    kind = rng.choices(("build", "host", "batch", "bounds"), (7, 1, 1, 1))[0]
    # grids and threshold go together: a threshold far below a grid layer's cells keeps nearly every
    # point on several levels, more than an output sized for such clouds holds
    chunking, subsampling, threshold = rng.choice(((512, 128, 10000), (512, 128, 10000), (256, 64, 5000),
                                                   (128, 64, 5000), (64, 32, 2000)))
    build = {"chunking_grid": chunking, "subsampling_grid": subsampling, "threshold": threshold,
             "filter": rng.choice(FILTERS), "explicit": rng.random() < 0.5, "output_factor": 4.0}
    if kind == "batch":
        least = _log(rng, 5_000, 40_000)
        build["filter"] = rng.choice(("none", "intra", "inter"))
        return {"kind": kind, "clouds": rng.randint(5, 64), "least": least, "most": least * rng.randint(3, 12), **build}
    dtype = rng.choice(("f32", "f64"))
    side = math.exp(rng.uniform(math.log(10.0), math.log(2000.0)))
    cloud = _cloud(_log(rng, 30_000, {"build": 40_000_000, "host": 4_000_000, "bounds": 100_000_000}[kind]) | 1, dtype,
                   side, side * rng.uniform(0.07, 0.6), rng.randint(2, 64), side * rng.uniform(0.004, 0.02),
                   0.0 if dtype == "f32" else 1e6)
    return {"kind": kind, **cloud} if kind == "bounds" else {"kind": kind, **cloud, **build}


def _members(case):
    """(points, record type) of a batch's clouds: sizes spread over their logarithm, large and small
    ones and the two types mixed."""
    count, ratio = case["clouds"], case["most"] / case["least"]
    sizes = [int(case["least"] * ratio ** ((i + 0.5) / count)) for i in range(count)]
    return [(sizes[i * 37 % count] if math.gcd(37, count) == 1 else sizes[i], ("f32", "f64")[i // 2 % 2])
            for i in range(count)]


# ---- what a program has in hand before the call -------------------------------------------------

def _make_cloud(case, seed):
    """The packed records (3 coordinates, RGB) of the case's cloud, in HBM."""
    device = torch.device("cuda", 0)
    gen = torch.Generator(device=device)
    gen.manual_seed(int(seed) * 2654435761 % (1 << 62))

    def rand(*shape):
        return torch.rand(*shape, generator=gen, device=device, dtype=torch.float64)

    n, dtype, side, height, clusters = case["points"], case["dtype"], case["side"], case["height"], case["clusters"]
    size = torch.float32 if dtype == "f32" else torch.float64
    amp, fx, fy, phase = 0.04 + 0.07 * rand(4), 0.5 + 3.5 * rand(4), 0.5 + 3.5 * rand(4), 2 * math.pi * rand(4)
    box = torch.tensor([side, side, height], device=device, dtype=torch.float64) * (0.9 + 0.1 * rand(3))
    centres = rand(clusters, 3) * box
    out = torch.empty(n, STRIDE[dtype], device=device, dtype=torch.uint8)
    for first in range(0, n, 1 << 23):
        m = min(1 << 23, n - first)
        uv = rand(m, 2)
        wave = torch.full((m,), 0.5, device=device, dtype=torch.float64)
        for j in range(4):
            wave += amp[j] * torch.sin(2 * math.pi * (fx[j] * uv[:, 0] + fy[j] * uv[:, 1]) + phase[j])
        field = torch.cat([uv, wave.unsqueeze(1)], 1) * box
        spread = torch.randn(m, 3, generator=gen, device=device, dtype=torch.float64) * case["sigma"]
        member = torch.randint(clusters, (m,), generator=gen, device=device)
        xyz = torch.where(rand(m, 1) < 0.7, field, centres[member] + spread)
        xyz = torch.minimum(torch.clamp(xyz, min=0.0), box)
        h = (xyz[:, 2] / height).unsqueeze(1)  # a height colour map with noise
        rgb = 255.0 * torch.cat([h, 1.0 - (2.0 * h - 1.0).abs(), 1.0 - h], 1)
        rgb += torch.randint(-16, 17, (m, 3), generator=gen, device=device)
        coords = (xyz + case["offset"]).to(size).contiguous().view(torch.uint8).reshape(m, -1)
        out[first:first + m, :coords.shape[1]] = coords
        out[first:first + m, coords.shape[1]:] = torch.clamp(rgb, 0, 255).to(torch.uint8)
    return out


def _bounding_box(cloud, dtype):
    real, cubic = np.zeros(6), np.zeros(6)
    rc = api.library().ocpi_compute_bounding_box(cloud.data_ptr(), cloud.shape[0], cloud.shape[1], CLOUD_TYPE[dtype], 0,
                                                 ctypes.c_void_p(real.ctypes.data), ctypes.c_void_p(cubic.ctypes.data))
    if rc != 0:
        raise api.OctreeError(api.last_error())
    return real, cubic


def _configured(case, cloud, seed):
    """A session with its cloud (in HBM) and configuration set."""
    dtype = case["dtype"]
    torch.cuda.synchronize()  # the cloud is complete before the library's own streams read it
    cubic = [float(v) for v in _bounding_box(cloud, dtype)[1]]
    session = api.Session(0)
    session.set_cloud(cloud, cloud.shape[0], cloud.shape[1], CLOUD_TYPE[dtype], cubic, [SCALE[dtype]] * 3,
                      device_pointer=cloud.data_ptr())
    color = case["filter"]
    session.configure(BuildSpec(case["chunking_grid"], case["threshold"], case["output_factor"],
                                case["subsampling_grid"], intra=color == "intra", inter=color in ("inter", "weighted"),
                                weighted=color == "weighted", random=case["explicit"], seed=int(seed)))
    return session, cubic


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        rng = np.random.default_rng(int(seed))
        sessions = []
        for i, (n, dtype) in enumerate(_members(case)):
            side = float(np.exp(rng.uniform(0.0, math.log(1000.0))))
            one = {**case, **_cloud(n, dtype, side, side * 0.2, int(rng.integers(2, 12)), side * 0.01,
                                    0.0 if dtype == "f32" else 1e5)}
            sessions.append(_configured(one, _make_cloud(one, seed * 1000 + i), seed)[0])
        return {"kind": kind, "builder": api.BatchBuilder(0), "sessions": sessions}
    cloud = _make_cloud(case, seed)
    if kind == "bounds":
        torch.cuda.synchronize()
        return {"kind": kind, "cloud": cloud, "dtype": case["dtype"]}
    session, cubic = _configured(case, cloud, seed)
    weighted = case["filter"] == "weighted"
    if kind == "host":
        return {"kind": kind, "session": session, "cloud": cloud.reshape(-1).cpu().numpy(), "points": case["points"],
                "dtype": case["dtype"], "cubic": cubic, "weighted": weighted}
    session.init()
    return {"kind": kind, "session": session, "weighted": weighted}


# ---- one pass -----------------------------------------------------------------------------------

class Octrees(dict):
    """The octrees that a pass has built, their nodes and records one after another. They stay where
    the pass left them (in HBM after a build) until a field is asked for, as with any program that
    builds now and exports later."""

    FIELDS = ("key", "count", "point_count", "data_idx", "parent", "children", "flags", "lut", "positions", "colors")

    def __init__(self, read, weighted=False):
        """read: a function that returns [(summary, nodes, lut, records)] of the octrees."""
        super().__init__((name, None) for name in self.FIELDS)
        self._read, self._fields, self._colors = read, None, torch.float16 if weighted else torch.int16

    def __getitem__(self, name):
        if self._fields is None:
            parts = [self._ordered(*octree, self._colors) for octree in self._read()]
            self._fields = {f: torch.cat([p[f] for p in parts]) if len(parts) > 1 else parts[0][f] for f in self.FIELDS}
        return self._fields[name]

    @staticmethod
    def _ordered(summary, nodes, lut, records, color_type):
        def padded(values, length, dtype):
            whole = torch.zeros(length, *values.shape[1:], device="cuda", dtype=dtype)
            whole[:len(values)] = values
            return whole

        fields = {f: torch.from_numpy(np.ascontiguousarray(getattr(nodes, f)).astype(np.int64)).cuda()
                  for f in Octrees.FIELDS[:7]}
        # the finished nodes' ranges tile the records: node by node, ascending point index
        held = ((fields["flags"] & 1) != 0) & (fields["point_count"] > 0)
        first, sizes = fields["data_idx"][held], fields["point_count"][held]
        node = torch.repeat_interleave(torch.arange(first.numel(), device="cuda"), sizes[torch.argsort(first)])
        lut, order = torch.sort((node << 32) | torch.from_numpy(lut.astype(np.int64)).cuda())
        raw = torch.from_numpy(records.view(np.uint8).reshape(-1, records.dtype.itemsize)).cuda()
        positions = torch.zeros(summary["capacity"], 3, device="cuda", dtype=torch.int32)
        colors = torch.zeros(summary["capacity"], 3, device="cuda", dtype=color_type)
        for at in range(0, len(records), 1 << 24):
            part = raw[order[at:at + (1 << 24)]]
            positions[at:at + len(part)] = part[:, :12].contiguous().view(torch.int32)
            colors[at:at + len(part)] = part[:, 12:].contiguous().view(torch.int16)
        most = min(summary["dense_nodes"], (summary["depth"] + 1) * summary["points"])
        return {**{f: padded(v, most, torch.int32) for f, v in fields.items()},
                "lut": padded(lut & 0xFFFFFFFF, summary["capacity"], torch.int32), "positions": positions,
                "colors": colors}


def _copied(session):
    summary = session.summary()
    return summary, session.nodes(), session.point_lut(summary["used"]), session.output(summary["used"])


def run(state):
    kind = state["kind"]
    if kind == "bounds":
        real, cubic = _bounding_box(state["cloud"], state["dtype"])
        return {"real": real, "cubic": cubic}
    if kind == "batch":
        state["builder"].build(state["sessions"])
        return Octrees(lambda: [_copied(s) for s in state["sessions"]])
    session = state["session"]
    if kind == "host":
        dtype = state["dtype"]
        session.set_cloud(state["cloud"], state["points"], STRIDE[dtype], CLOUD_TYPE[dtype], state["cubic"],
                          [SCALE[dtype]] * 3)
        session.init()
        session.generate()
        octree = _copied(session)
        return Octrees(lambda: [octree], state["weighted"])
    session.generate()
    return Octrees(lambda: [_copied(session)], state["weighted"])


def work(case):
    """The records read once; the octree's records and point indices written once. A build does no
    contraction, and its cell mappings are a few operations a point, so no operations are counted."""
    if case["kind"] == "batch":
        return {"bytes": sum(n * (STRIDE[t] + 22 * RECORDS_PER_POINT) for n, t in _members(case)), "flops": 0}
    points, stride = case["points"], STRIDE[case["dtype"]]
    if case["kind"] == "bounds":
        return {"bytes": points * (stride - 3), "flops": 0}  # the coordinates
    return {"bytes": points * (stride + 22 * RECORDS_PER_POINT), "flops": 0}


# ---- exact values -------------------------------------------------------------------------------

def _records(cloud, dtype):
    """(coordinates in 64 bits, colours) of packed records."""
    width, size = (4, torch.float32) if dtype == "f32" else (8, torch.float64)
    parts = [cloud[at:at + (1 << 24), :3 * width].contiguous().view(size).double() for at in range(0, len(cloud), 1 << 24)]
    return torch.cat(parts), cloud[:, 3 * width:]


def _box(xyz):
    """The real bounding box and the cube around it."""
    least, most = xyz.amin(0).cpu().numpy(), xyz.amax(0).cpu().numpy()
    side = (most - least).max()
    corner = least - (side - (most - least)) / 2.0
    return np.concatenate([least, most]), np.concatenate([corner, corner + side])


def _ranks(index, node, salt_of, explicit):
    """The order in which points of a node are preferred: by index, or by a hash of it keyed by the node."""
    if not explicit:
        return index
    values, inverse = torch.unique(node, return_inverse=True)
    h = index ^ torch.tensor([salt_of(int(v)) for v in values], device=index.device)[inverse]
    for shift, factor in ((16, 0x85EBCA6B), (13, 0xC2B2AE35), (16, 1)):
        h = ((h ^ (h >> shift)) * factor) & 0xFFFFFFFF
    return h


def _weighted_colors(case, seed):
    """The colours of a build with the distance-weighted filter: the octree level by level, bottom
    up, every average in 64 bits (and then cut to whole numbers, as a record holds it)."""
    xyz, rgb = _records(_make_cloud(case, seed), case["dtype"])
    cubic = _box(xyz)[1]
    n, grid, g, threshold = len(xyz), case["chunking_grid"], case["subsampling_grid"], case["threshold"]
    depth, size = grid.bit_length() - 1, float(cubic[3] - cubic[0])
    least = torch.from_numpy(cubic[:3]).cuda()
    cell = torch.clamp((xyz - least) / (size / grid), max=grid - 1.0).long()
    every = torch.arange(n, device="cuda")

    def linear(at, level):
        side, c = grid >> level, cell[at] >> level
        return c[:, 0] + c[:, 1] * side + c[:, 2] * side * side

    def morton(c, bits):
        code = torch.zeros_like(c[:, 0])
        for b in range(bits):
            for axis, to in ((0, 2), (1, 1), (2, 0)):
                code |= ((c[:, axis] >> b) & 1) << (3 * b + to)
        return code

    # the level of every point's leaf: the lowest whose parent holds at least `threshold` points
    leaf = torch.full((n,), depth, device="cuda")
    for level in range(depth, 0, -1):
        at = linear(every, level)
        leaf = torch.where(torch.bincount(at, minlength=(grid >> level) ** 3)[at] >= threshold, level - 1, leaf)
    # leaf blocks lie in the order of their parents (level, then cell), in slot order inside
    place = torch.zeros(n, device="cuda", dtype=torch.int64)
    for level in range(depth):
        at = torch.nonzero(leaf == level).squeeze(1)
        slot = (cell[at] >> level) & 1
        place[at] = (((level << 32) + linear(at, level + 1)) << 3) + 4 * slot[:, 0] + 2 * slot[:, 1] + slot[:, 2]
    colors = [rgb[torch.sort(place, stable=True)[1]].double()]

    inner, offset = [], 0
    index, color = every[:0], colors[0][:0]
    for level in range(1, depth + 1):
        offset += (grid >> (level - 1)) ** 3  # of the level's cells among all dense cells
        more = torch.nonzero(leaf == level - 1).squeeze(1)
        index, color = torch.cat([index, more]), torch.cat([color, rgb[more].double()])
        if len(index) == 0:
            continue
        node_cell = cell[index] >> level
        corner = least.expand(len(index), 3).clone()
        for up in range(depth, level, -1):
            corner += ((node_cell >> (up - 1 - level)) & 1).double() * (size / 2.0 ** (depth - up) / 2.0)
        side = size / 2.0 ** (depth - level)
        t = ((corner[:, :1] + side) - corner[:, :1]) / g
        inside = torch.clamp((xyz[index] - corner) / t, max=g - 1.0).long()
        node = linear(index, level)
        key = node * g ** 3 + inside[:, 0] + inside[:, 1] * g + inside[:, 2] * g * g
        cells, member = torch.unique(key, return_inverse=True)

        def salt_of(v):
            z, mask = (int(seed) + 0x9E3779B97F4A7C15 * (offset + v + 1)) & (2 ** 64 - 1), 2 ** 64 - 1
            z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & mask
            z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & mask
            return (z ^ (z >> 31)) >> 32

        # a 32-bit rank, kept in the sign's range, then the index that it names
        rank = ((_ranks(index, node, salt_of, case["explicit"]) - 2 ** 31) << 32) | index
        winner = torch.full((len(cells),), 2 ** 63 - 1, device="cuda")
        winner.scatter_reduce_(0, member, rank, "amin")
        total = torch.zeros(len(cells), 4, device="cuda", dtype=torch.float64)
        what = torch.cat([color, torch.ones_like(color[:, :1])], 1)
        reach = (t * 3) ** 2 * 3 / 4.0  # half the diagonal of three cells, squared
        for step in range(27):
            d = torch.tensor([step % 3 - 1, step // 3 % 3 - 1, step // 9 - 1], device="cuda")
            to = inside + d
            wanted = key + int(d[0] + d[1] * g + d[2] * g * g)
            found = torch.searchsorted(cells, wanted).clamp(max=len(cells) - 1)
            hit = ((to >= 0) & (to < g)).all(1) & (cells[found] == wanted)
            away = (corner + to * t + t * 0.5 - xyz[index])[hit]
            weight = torch.exp(-10.0 * (away * away).sum(1, keepdim=True) / reach[hit])
            total.index_add_(0, found[hit], what[hit] * weight)
        index, color = winner & 0xFFFFFFFF, torch.floor(total[:, :3] / total[:, 3:])
        end = (morton(cell[index] >> level, depth - level) + 1) << (3 * level)  # of the node's range: post-order
        inner.append((((end << 4) + level) << 28 | index, color))  # 31 bits, and at most 30 million points
    if inner:
        order = torch.sort(torch.cat([k for k, _ in inner]))[1]
        colors.append(torch.cat([c for _, c in inner])[order])
    capacity = int(np.float32(n) * np.float32(case["output_factor"]))
    colors.append(torch.zeros(capacity - sum(len(c) for c in colors), 3, device="cuda", dtype=torch.float64))
    return torch.cat(colors)


def exact(case, seed):
    """A bounding box and the distance-weighted colours; all else of an octree is whole numbers."""
    if case["kind"] == "bounds":
        real, cubic = _box(_records(_make_cloud(case, seed), case["dtype"])[0])
        return {"real": real, "cubic": cubic}
    if case["filter"] != "weighted" or case["points"] > 30_000_000:  # beyond that it takes too long
        return None
    return {**{name: None for name in Octrees.FIELDS}, "colors": _weighted_colors(case, seed)}

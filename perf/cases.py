"""The work this framework is measured on: what a user of sparse convolutions
has it do, through its public entry points.

Kinds of case

* ``voxelize``: raw points to voxels, the first thing done with every scan.
* ``map``: the Map step alone, unsorted voxels to sorted voxels and per-offset
  pair lists.
* ``conv``: one layer on a tensor whose kernel map its cache already holds, as
  every layer but the first of a level sees it (configurations 1, 2 and 5).
* ``downup``: a strided layer and its transposed twin on a new cloud: strided
  coordinates, kernel map and both directions (configuration 3).
* ``unet`` / ``resnet``: a whole network on a new batch of unsorted clouds:
  collating, every kernel map, every layer (configuration 4).

Clouds are surfaces, because that is what sensors see: ``lidar`` (a rotating
scanner over ground and boxes), ``room`` (walls and furniture) and ``object``
(tilted planes and spheres).  They are generated on the GPU from the seed, with
the densities of the generators in ``minuet_amd.synthetic``.
"""
import functools
import math

import numpy as np
import torch

import minuet_amd as minuet
from minuet_amd.nn import functional as F
from minuet_amd.nn.functional import _C
from minuet_amd.resnet import SparseResNet
from minuet_amd.unet import SparseUNet
from minuet_amd.utils.helpers import generate_kernel_offsets

DTYPES = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}


def listed():
    return [
        # one scan of a spinning scanner, a little over 64 rings x 2048 azimuths less the sky
        {"name": "voxelize lidar 100k", "kind": "voxelize", "scene": "lidar", "points": 100003},
        # the smallest call: one scanned object, launches and latency
        {"name": "map object 2k", "kind": "map", "scene": "object", "voxels": 2039, "kernel": 3},
        # configuration 2
        {"name": "map lidar 200k", "kind": "map", "scene": "lidar", "voxels": 200000, "kernel": 3},
        # configuration 1: fp32, the reference's own feature type
        {"name": "conv object 20k fp32", "kind": "conv", "scene": "object", "voxels": 20000, "kernel": 3,
         "dilation": 1, "cin": 32, "cout": 32, "dtype": "fp32", "bias": False},
        # a wider fp32 layer of an odd-sized cloud, with a bias, channels no power of two
        {"name": "conv room 61k fp32 wide", "kind": "conv", "scene": "room", "voxels": 61057, "kernel": 3,
         "dilation": 1, "cin": 64, "cout": 96, "dtype": "fp32", "bias": True},
        # the 64-channel fp16 layer on the configuration-2 cloud
        {"name": "conv lidar 200k fp16", "kind": "conv", "scene": "lidar", "voxels": 200000, "kernel": 3,
         "dilation": 1, "cin": 64, "cout": 64, "dtype": "fp16", "bias": False},
        # the wide layers of a network's coarse levels
        {"name": "conv lidar 26k fp16 wide", "kind": "conv", "scene": "lidar", "voxels": 25641, "kernel": 3,
         "dilation": 1, "cin": 256, "cout": 256, "dtype": "fp16", "bias": False},
        # configuration 5: large kernel, a million voxels
        {"name": "conv lidar 1m bf16 k5", "kind": "conv", "scene": "lidar", "voxels": 1000000, "kernel": 5,
         "dilation": 1, "cin": 64, "cout": 64, "dtype": "bf16", "bias": False},
        # configuration 3
        {"name": "downup room 150k fp16", "kind": "downup", "scene": "room", "voxels": 150000,
         "cin": 64, "cout": 128, "dtype": "fp16"},
        # configuration 4
        {"name": "unet lidar 2x100k fp16", "kind": "unet", "scene": "lidar", "voxels": 100000, "batch": 2,
         "dtype": "fp16"},
        # a small cloud in the reference's feature type, one at a time
        {"name": "unet room 1x12k fp32", "kind": "unet", "scene": "room", "voxels": 12007, "batch": 1,
         "dtype": "fp32"},
        # classification of a batch of small objects
        {"name": "resnet object 8x3k bf16", "kind": "resnet", "scene": "object", "voxels": 3001, "batch": 8,
         "dtype": "bf16"},
    ]


def _between(rng, low, high):
    """A whole number from ``low`` to ``high``, spread over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["voxelize", "map", "map", "conv", "conv", "conv", "conv", "downup", "unet", "resnet"])
    scene = rng.choice(["lidar", "room", "object"])
    dtype = rng.choice(["fp16", "fp16", "bf16", "fp32"])
    if kind == "voxelize":
        return {"kind": kind, "scene": scene, "points": _between(rng, 2000, 1000000)}
    if kind == "map":
        return {"kind": kind, "scene": scene, "voxels": _between(rng, 1000, 1000000),
                "kernel": rng.choice([3, 3, 3, 5])}
    if kind == "conv":
        kernel = rng.choice([3, 3, 3, 5])
        cin = rng.choice([3, 4, 16, 24, 32, 48, 64, 96, 128, 192, 256])
        cout = rng.choice([16, 32, 48, 64, 96, 128, 256])
        # no more multiply-adds than the million-voxel layer; fp32 ones are that much dearer on the matrix cores
        most = 1.0e6 * 125 * 64 * 64 / (16.0 if dtype == "fp32" else 2.0) / (kernel ** 3 * cin * cout)
        return {"kind": kind, "scene": scene, "voxels": _between(rng, 1000, min(1000000, max(2000, int(most)))),
                "kernel": kernel, "dilation": rng.choice([1, 1, 1, 2]), "cin": cin, "cout": cout,
                "dtype": dtype, "bias": rng.random() < 0.3}
    if kind == "downup":
        cin = rng.choice([16, 32, 64, 128])
        return {"kind": kind, "scene": scene, "voxels": _between(rng, 2000, 300000), "cin": cin,
                "cout": rng.choice([cin, 2 * cin]), "dtype": dtype}
    batch = rng.choice([1, 1, 2, 3, 4, 8])
    most = 12000 if dtype == "fp32" else 180000
    return {"kind": kind, "scene": scene, "voxels": _between(rng, 1000, most // batch), "batch": batch,
            "dtype": dtype}


# ------------------------------------------------------------------ clouds ----

_DEVICE = torch.device("cuda:0")
_HALF = 1 << 19          # coordinates lie in [-_HALF, _HALF)


def _uniform(gen, shape, low=0.0, high=1.0):
    return torch.rand(shape, generator=gen, device=_DEVICE, dtype=torch.float64) * (high - low) + low


def _lidar_points(gen, sweeps, trajectory):
    """Hits of ``sweeps`` revolutions of a 64-ring scanner 1.8 m over the ground
    among 30 boxes (the same boxes for every call with the same seed)."""
    where = 50.0 * torch.sqrt(_uniform(gen, (30,)))
    angle = _uniform(gen, (30,), 0.0, 2.0 * math.pi)
    size = torch.stack([_uniform(gen, (30,), 1, 6), _uniform(gen, (30,), 1, 6), _uniform(gen, (30,), 1, 4)], 1)
    centre = torch.stack([where * torch.cos(angle), where * torch.sin(angle), size[:, 2] / 2], 1)
    low, high = centre - size / 2, centre + size / 2
    near = ((low[:, :2] < 1.5) & (high[:, :2] > -1.5)).all(1, keepdim=True)
    low, high = low + 1e6 * near, high + 1e6 * near          # no box around the scanner
    elevation = torch.linspace(-24.8, 2.0, 64, device=_DEVICE, dtype=torch.float64) * (math.pi / 180.0)
    chunks = []
    for s in range(sweeps):
        jitter = _uniform(gen, (3,), -1.0, 1.0)
        along = trajectory * ((s * 0.25 / max(trajectory, 0.25)) % 1.0 - 0.5) if trajectory > 0 else 0.0
        at = torch.stack([0.5 * jitter[0] + along, 0.5 * jitter[1], torch.full_like(jitter[0], 1.8)])
        azimuth = jitter[2] * math.pi / 2048 + torch.arange(2048, device=_DEVICE) * (2.0 * math.pi / 2048)
        flat = torch.cos(elevation)[:, None]
        ray = torch.stack([flat * torch.cos(azimuth), flat * torch.sin(azimuth),
                           torch.sin(elevation)[:, None].expand(64, 2048)], -1).reshape(-1, 3)
        best = torch.where(ray[:, 2] < -1e-9, -at[2] / ray[:, 2], torch.inf)
        a, b = (low - at) / ray[:, None], (high - at) / ray[:, None]
        enter, leave = torch.minimum(a, b).amax(2), torch.maximum(a, b).amin(2)
        hit = torch.where((leave >= enter) & (enter > 1e-6), enter, torch.inf).amin(1)
        best = torch.minimum(best, hit)
        keep = best <= 50.0
        chunks.append(at + ray[keep] * best[keep, None])
    return torch.cat(chunks)


def _room_points(gen, count):
    """Samples of the walls of an 8 x 6 x 3 m room and of 40 boxes in it."""
    room = torch.tensor([8.0, 6.0, 3.0], device=_DEVICE, dtype=torch.float64)
    extent = torch.cat([room[None], _uniform(gen, (40, 3), 0.2, 1.5)])
    corner = torch.zeros_like(extent)
    corner[1:, :2] = _uniform(gen, (40, 2)) * (room[:2] - extent[1:, :2])
    area = torch.stack([extent[:, 1] * extent[:, 2], extent[:, 0] * extent[:, 2], extent[:, 0] * extent[:, 1]], 1)
    share = torch.full((41,), 0.3 / 40, device=_DEVICE, dtype=torch.float64)
    share[0] = 0.7
    body = torch.bucketize(_uniform(gen, (count,)), torch.cumsum(share, 0)[:-1])
    edges = torch.cumsum(area / area.sum(1, keepdim=True), 1)[body]
    pick = _uniform(gen, (count, 1))
    axis = (pick > edges[:, :2]).sum(1)
    inside = _uniform(gen, (count, 3))
    side = torch.randint(0, 2, (count,), generator=gen, device=_DEVICE).double() * (1.0 - 1e-9)
    inside.scatter_(1, axis[:, None], side[:, None])
    return torch.minimum(corner[body] + inside * extent[body], room - 1e-6)


def _object_points(gen, count):
    """Samples of four tilted planes and two spheres in the unit cube."""
    chunks = []
    for _ in range(4):
        normal = torch.nn.functional.normalize(torch.randn(3, generator=gen, device=_DEVICE).double(), dim=0)
        u = torch.linalg.cross(normal, torch.roll(normal, 1))
        u = torch.nn.functional.normalize(u, dim=0)
        v = torch.linalg.cross(normal, u)
        ab = _uniform(gen, (count // 3, 2), -1.0, 1.0)
        chunks.append(_uniform(gen, (3,), 0.25, 0.75) + ab[:, :1] * u + ab[:, 1:] * v)
    for _ in range(2):
        way = torch.nn.functional.normalize(torch.randn(count // 3, 3, generator=gen, device=_DEVICE).double(), dim=1)
        chunks.append(_uniform(gen, (3,), 0.25, 0.75) + _uniform(gen, (1,), 0.1, 0.25) * way)
    points = torch.cat(chunks)
    return points[((points >= 0) & (points < 1)).all(1)]


def _pack(voxels):
    v = voxels.long() + _HALF
    return (v[:, 0] << 40) | (v[:, 1] << 20) | v[:, 2]


def _unpack(keys):
    return torch.stack([(keys >> 40) & 0xFFFFF, (keys >> 20) & 0xFFFFF, keys & 0xFFFFF], 1) - _HALF


def _generator(seed):
    gen = torch.Generator(device=_DEVICE)
    gen.manual_seed(int(seed) & 0x7FFFFFFF)
    return gen


def _points(scene, count, seed):
    """``(points, voxel size)``: at least as many surface points as voxels of
    that size are wanted; small clouds have coarser voxels, as they have in use."""
    if scene == "lidar":
        sweeps = max(1, -(-count // 30000))
        points = _lidar_points(_generator(seed), sweeps, 20.0 if count > 400000 else 0.0)
        return points, 0.05 * max(1.0, math.sqrt(60000.0 / count))
    if scene == "room":
        return _room_points(_generator(seed), int(2.2 * count) + 1024), 0.02 * math.sqrt(150000.0 / count)
    return _object_points(_generator(seed), int(1.6 * count) + 1024), math.sqrt(20000.0 / count) / 128.0


def _another_view(voxels, gen):
    """The same voxels from another heading and place: x and y flipped and
    swapped, everything moved.  How many neighbours they have stays what it was."""
    flips = torch.randint(0, 2, (3,), generator=gen, device=_DEVICE).tolist()
    x, y, z = voxels.unbind(1)
    x, y = (-1 - x if flips[0] else x), (-1 - y if flips[1] else y)
    turned = torch.stack([y, x, z] if flips[2] else [x, y, z], 1)
    return turned + torch.randint(-500, 500, (3,), generator=gen, device=_DEVICE)


def _cloud(scene, count, seed):
    """Exactly ``count`` distinct voxels [count, 3] int32 in no particular order."""
    wanted = count
    while True:
        points, size = _points(scene, wanted, seed)
        keys = torch.unique(_pack(torch.floor(points / size)))
        if keys.shape[0] >= count:
            break
        wanted = int(1.3 * wanted) + 64
    gen = _generator(seed + 77)
    keep = torch.randperm(keys.shape[0], generator=gen, device=_DEVICE)[:count]
    return _unpack(keys[keep]).to(torch.int32).contiguous()


# ----------------------------------------------------------- states, passes ----

def _features(rows, channels, dtype, seed):
    return torch.randn(rows, channels, generator=_generator(seed + 5), device=_DEVICE).to(DTYPES[dtype])


def _network(case, seed):
    torch.manual_seed(int(seed) & 0x7FFFFFFF)
    factory = {"dtype": DTYPES[case["dtype"]], "device": _DEVICE}
    net = SparseUNet(4, 32, **factory) if case["kind"] == "unet" else SparseResNet(4, 10, **factory)
    gen = _generator(seed + 9)
    with torch.no_grad():
        for module in net.modules():         # a trained network's statistics and weights, not those of an untouched one
            if isinstance(module, minuet.nn.SparseConv):
                fan = module.in_channels * max(1.0, module.kernel.shape[0] * 0.3)
                module.kernel.normal_(0.0, math.sqrt(2.0 / fan), generator=gen)
            elif isinstance(module, minuet.nn.BatchNorm):
                module.running_mean.uniform_(-0.2, 0.2, generator=gen)
                module.running_var.uniform_(0.8, 1.5, generator=gen)
    return net.eval()


def _new_cache(*modules):
    cache = minuet.nn.KernelMapCache(3, torch.int32, _DEVICE)
    for module in modules:
        minuet.set_kernel_map_cache(module, cache)
    return cache


@torch.no_grad()
def prepare(case, seed):
    kind = case["kind"]
    if kind in ("voxelize", "map"):
        # The lengths of these results depend on the scene, so it is one scene of
        # that size for every seed: seen from another side, in another order.
        gen = _generator(seed)
        if kind == "map":
            offsets = np.ascontiguousarray(generate_kernel_offsets(3, case["kernel"], 1, 1), dtype=np.int64)
            voxels = _another_view(_cloud(case["scene"], case["voxels"], 4242).long(), gen)
            order = torch.randperm(case["voxels"], generator=gen, device=_DEVICE)
            return kind, voxels[order].to(torch.int32).contiguous(), offsets
        points, size = _points(case["scene"], case["points"], 4242)
        while points.shape[0] < case["points"]:
            points = torch.cat([points, points])
        pick = torch.randperm(points.shape[0], generator=_generator(4242), device=_DEVICE)[:case["points"]]
        voxels = _another_view(torch.floor(points[pick] / size).long(), gen)
        order = torch.randperm(case["points"], generator=gen, device=_DEVICE)
        points = (voxels[order] + _uniform(gen, (case["points"], 3), 0.02, 0.98)) * size
        return kind, points.float().contiguous(), size
    if kind in ("conv", "downup"):
        voxels = _cloud(case["scene"], case["voxels"], seed)
        coordinates = voxels[F.build_sorted_index(voxels)]
        features = _features(case["voxels"], case["cin"], case["dtype"], seed)
        factory = {"dtype": DTYPES[case["dtype"]], "device": _DEVICE}
        torch.manual_seed(int(seed) & 0x7FFFFFFF)
        if kind == "downup":
            down = minuet.nn.SparseConv3d(case["cin"], case["cout"], 2, stride=2, **factory)
            up = minuet.nn.SparseConv(3, case["cout"], case["cin"], 2, stride=2, transposed=True, **factory)
            return kind, coordinates, features, down, up, _new_cache(down, up)
        conv = minuet.nn.SparseConv3d(case["cin"], case["cout"], case["kernel"], dilation=case["dilation"],
                                      bias=case["bias"], **factory)
        cache = _new_cache(conv)
        x = minuet.SparseTensor(features, coordinates)
        conv(x)                              # the level's first layer: leaves its kernel map in the cache
        return kind, x, conv, cache
    clouds = [_cloud(case["scene"], case["voxels"], seed + 1000 * b) for b in range(case["batch"])]
    features = [_features(case["voxels"], 4, case["dtype"], seed + 1000 * b) for b in range(case["batch"])]
    net = _network(case, seed)
    return kind, clouds, features, net, _new_cache(net)


@torch.no_grad()
def run(state):
    kind = state[0]
    if kind == "voxelize":
        return F.voxelize(state[1], voxel_size=state[2], return_reverse_indices=True)
    if kind == "map":
        built = _C.sorted_kernel_map_lists(state[1], state[2], reorder=True, result_only=True)
        return [built[name] for name in ("indices", "coordinates", "in_idx", "out_idx", "sizes_host", "order_host")]
    if kind == "conv":
        return state[2](state[1]).F
    if kind == "downup":
        _, coordinates, features, down, up, cache = state
        cache.reset()
        low = down(minuet.SparseTensor(features, coordinates))
        high = up(low)
        return high.C, high.F
    _, clouds, features, net, cache = state
    coordinates, batch_dims, rows = F.collate(clouds, features)
    cache.reset()
    result = net(minuet.SparseTensor(rows, coordinates, batch_dims=batch_dims))
    return (result.C, result.F) if kind == "unet" else result


# ------------------------------------------------------- what a pass must do ----

def _bytes_of(dtype):
    return DTYPES[dtype].itemsize


def _hits(sources, targets, kernel, spacing):
    """Hits of a kernel map between two sorted arrays of packed keys."""
    offsets = torch.from_numpy(np.ascontiguousarray(generate_kernel_offsets(3, kernel, spacing, 1))).long()
    total = 0
    for x, y, z in offsets.tolist():
        wanted = targets + ((x << 40) + (y << 20) + z)
        at = torch.searchsorted(sources, wanted).clamp_(max=sources.shape[0] - 1)
        total += int((sources[at] == wanted).sum())
    return total


def _coarser(keys, stride):
    batch = keys >> 60
    v = torch.div(_unpack(keys), stride, rounding_mode="floor") * stride
    return torch.unique(_pack(v) | (batch << 60))


@functools.lru_cache(maxsize=64)
def _levels(scene, voxels, batch, levels):
    """Per level of a batch of typical clouds: (voxels, hits of 3x3x3)."""
    keys = torch.sort(torch.cat([_pack(_cloud(scene, voxels, 4242 + 1000 * b)) | (b << 60)
                                 for b in range(batch)]))[0]
    found = []
    for level in range(levels):
        if level:
            keys = _coarser(keys, 2 ** level)
        found.append((keys.shape[0], _hits(keys, keys, 3, 2 ** level)))
    return found


@functools.lru_cache(maxsize=64)
def _layer_hits(scene, voxels, kernel, spacing):
    keys = torch.sort(_pack(_cloud(scene, voxels, 4242)))[0]
    return _hits(keys, keys, kernel, spacing)


def _layer(rows_in, rows_out, hits, volume, cin, cout, size):
    """(bytes, flops) of one layer: features in and out, weights and a source row per hit, once each."""
    return (size * (rows_in * cin + rows_out * cout + volume * cin * cout) + 4 * hits, 2 * hits * cin * cout)


def _network_layers(kind, levels):
    """(rows in, rows out, hits, volume, cin, cout) of every layer."""
    layers = []

    def blocks(level, cin, cout):
        n, hits = levels[level]
        layers.extend([(n, n, hits, 27, cin, cout)] + 3 * [(n, n, hits, 27, cout, cout)])
        if cin != cout:
            layers.append((n, n, n, 1, cin, cout))

    first, hits = levels[0]
    layers.append((first, first, hits, 27, 4, 32))
    widths = [32, 32, 64, 128, 256] if kind == "unet" else [32, 64, 128, 256]
    for level in range(1, len(widths)):
        fine, coarse = levels[level - 1][0], levels[level][0]
        layers.append((fine, coarse, fine, 8, widths[level - 1], widths[level]))
        blocks(level, widths[level], widths[level])
    if kind == "unet":
        current = 256
        for level, width in zip((3, 2, 1, 0), (128, 64, 32, 32)):
            layers.append((levels[level + 1][0], levels[level][0], levels[level][0], 8, current, width))
            blocks(level, width + widths[level], width)
            current = width
        layers.append((first, first, first, 1, 32, 32))
    return layers


def work(case):
    kind = case["kind"]
    if kind == "voxelize":           # points in, voxels (about half as many as points) and a row per point out
        return {"bytes": case["points"] * (12 + 8 + 6), "flops": 0}
    n = case["voxels"]
    if kind == "map":                # voxels in; permutation, sorted voxels and two list entries per hit out
        hits = _layer_hits(case["scene"], n, case["kernel"], 1)
        return {"bytes": n * (12 + 4 + 12) + 8 * hits, "flops": 0}
    size = _bytes_of(case["dtype"])
    if kind == "conv":
        hits = _layer_hits(case["scene"], n, case["kernel"], case["dilation"])
        nbytes, flops = _layer(n, n, hits, case["kernel"] ** 3, case["cin"], case["cout"], size)
        return {"bytes": nbytes, "flops": flops}
    if kind == "downup":             # the strided voxels are written and the map is one parent per voxel
        keys = torch.sort(_pack(_cloud(case["scene"], n, 4242)))[0]
        coarse = _coarser(keys, 2).shape[0]
        down = _layer(n, coarse, n, 8, case["cin"], case["cout"], size)
        up = _layer(coarse, n, n, 8, case["cout"], case["cin"], size)
        return {"bytes": down[0] + up[0] + 12 * (n + coarse), "flops": down[1] + up[1]}
    levels = _levels(case["scene"], n, case["batch"], 5 if kind == "unet" else 4)
    parts = [_layer(*layer, size) for layer in _network_layers(kind, levels)]
    collated = 2 * case["batch"] * n * (12 + 4 * size)
    return {"bytes": collated + sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}


def tolerance(case):
    """Voxels, permutations and lists are exact.  A layer sums in fp32 and rounds
    its output once (a three-kernel layer its products too); a network rounds
    after each of its 20 to 46 layers."""
    if case["kind"] in ("voxelize", "map"):
        return "exact"
    if case["kind"] in ("conv", "downup"):
        return {"rel": {"fp32": 1e-5, "fp16": 2e-3, "bf16": 1e-2}[case["dtype"]]}
    return {"rel": {"fp32": 1e-5, "fp16": 5e-3, "bf16": 2e-2}[case["dtype"]]}

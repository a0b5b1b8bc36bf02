"""Voxelisation, collating and global pools at the edges of their tiles."""
import numpy as np
import pytest
import torch

import minuet_oracle as orc
from helpers import dev, host, random_cloud, sorted_unique
from minuet_amd.nn import functional as F
from minuet_amd.nn.functional import _C
from minuet_amd.tensors import SparseTensor

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,ndim,ftype,dtype", [(1, 3, np.float32, torch.int32), (2049, 3, np.float64, torch.int64),
                                                (5000, 2, np.float32, torch.int32), (4096, 4, np.float32, torch.int64),
                                                (1049089, 3, np.float32, torch.int32)])
def test_voxelize_against_numpy(n, ndim, ftype, dtype):
    points = np.random.default_rng(n).normal(size=(n, ndim)).astype(ftype)
    size = tuple(0.11 + 0.07 * k for k in range(ndim))
    voxels, reverse = F.voxelize(dev(points), voxel_size=size, dtype=dtype, return_reverse_indices=True)
    expect, inverse = np.unique(np.floor(points / np.asarray(size, dtype=ftype)).astype(np.int64), axis=0,
                                return_inverse=True)
    assert voxels.dtype == dtype and reverse.dtype == torch.int64
    np.testing.assert_array_equal(host(voxels), expect)
    np.testing.assert_array_equal(host(reverse), inverse.reshape(-1))


@pytest.mark.parametrize("n,ndim,ftype,dtype", [(4097, 4, np.float64, torch.int64), (5121, 1, np.float32, torch.int32),
                                                (131073, 3, np.float64, torch.int32), (140001, 2, np.float32, torch.int64)])
def test_voxels_leave_their_bounds(n, ndim, ftype, dtype):
    """Clouds whose voxels and bounds come of one launch: one far corner in the last
    row, one in the first, coordinates of both signs, runs of equal points."""
    rng = np.random.default_rng(n)
    points = rng.integers(-40, 40, size=(n, ndim)).astype(ftype) + ftype(0.5)
    points[-1], points[0] = 3000.5, -2999.5
    voxels, reverse = F.voxelize(dev(points), voxel_size=1.0, dtype=dtype, return_reverse_indices=True)
    expect, inverse = np.unique(np.floor(points).astype(np.int64), axis=0, return_inverse=True)
    np.testing.assert_array_equal(host(voxels), expect)
    np.testing.assert_array_equal(host(reverse), inverse.reshape(-1))


@pytest.mark.parametrize("rows,channels", [((7,), 1), ((0, 3, 900), 6), ((5000, 1, 20000), 64), ((300, 41), 257),
                                           ((130,), 1100)])
@pytest.mark.parametrize("kind", ["fp32", "fp16", "bf16"])
def test_global_pools(rows, channels, kind):
    dtype = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}[kind]
    bounds = np.concatenate([[0], np.cumsum(rows)])
    n = int(bounds[-1])
    f = torch.randn(n, channels, device="cuda").to(dtype)
    c = dev(np.arange(3 * n, dtype=np.int32).reshape(n, 3))
    for itype in (np.int32, np.int64):
        x = SparseTensor(f, c, batch_dims=dev(bounds.astype(itype)))
        exact = f.double().cpu().numpy()
        for pool, fold in ((F.global_avg_pool, np.mean), (F.global_sum_pool, np.sum)):
            got = pool(x).double().cpu().numpy().reshape(len(rows), channels)
            for g, count in enumerate(rows):
                if count == 0:
                    assert np.isnan(got[g]).all() if fold is np.mean else (got[g] == 0).all()
                    continue
                part = exact[bounds[g]:bounds[g + 1]]
                want = fold(part, axis=0)
                eps = {"fp32": 1e-5, "fp16": 1e-3, "bf16": 8e-3}[kind]
                scale = np.abs(part).sum(axis=0) / (count if fold is np.mean else 1)
                assert (np.abs(got[g] - want) <= eps * np.abs(want) + 1e-6 * scale).all()


@pytest.mark.parametrize("channels,dtype", [(1, torch.float16), (4, torch.float16), (3, torch.float32), (8, torch.float32)])
@pytest.mark.parametrize("clouds", [1, 3, 70])
def test_collate_carries_rows(channels, dtype, clouds):
    coords = [sorted_unique(random_cloud(5 + 40 * (k % 3), 30, k))[0] for k in range(clouds)]
    feats = [torch.randn(c.shape[0], channels, device="cuda").to(dtype) for c in coords]
    ordered, dims, rows = F.collate([dev(c) for c in coords], feats)
    plain, plain_dims = F.collate([dev(c) for c in coords])
    bounds = np.concatenate([[0], np.cumsum([c.shape[0] for c in coords])])
    order = orc.arg_sort_coordinates(np.concatenate(coords), bounds.astype(np.int32))
    assert torch.equal(ordered, plain) and torch.equal(dims, plain_dims)
    np.testing.assert_array_equal(host(dims), bounds)
    assert torch.equal(rows, torch.cat(feats)[dev(order.astype(np.int64))])


# rows in all: one, the small sort's 4 096 and one more, a bucket sort's, and more than it takes; clouds
# without a row in front, between and behind; as many clouds as one call takes, and one more
@pytest.mark.parametrize("sizes,ndim,dtype", [
    ([1], 3, np.int32), ([0, 4091, 0, 5, 0], 3, np.int32), ([0, 4092, 5, 0], 4, np.int64), ([70] * 64, 2, np.int32),
    ([70] * 65, 2, np.int64), ([40000, 1, 30001], 1, np.int64), ([131073, 2], 3, np.int32), ([2100001], 3, np.int32)])
def test_collate_in_one_call(sizes, ndim, dtype):
    coords = [random_cloud(n, 1 << 20, k, ndim=ndim, lo=-(1 << 19), dtype=dtype) for k, n in enumerate(sizes)]
    feats = [torch.arange(3 * n, device="cuda", dtype=torch.float32).view(n, 3) - 7 * k for k, n in enumerate(sizes)]
    ordered, dims, rows = F.collate([dev(c) for c in coords], feats)
    bounds = np.concatenate([[0], np.cumsum(sizes)])
    order = orc.arg_sort_coordinates(np.concatenate(coords), bounds.astype(dtype) if len(sizes) > 1 else None)
    assert ordered.dtype == dims.dtype == torch.from_numpy(coords[0]).dtype
    np.testing.assert_array_equal(host(ordered), np.concatenate(coords)[order])
    np.testing.assert_array_equal(host(dims), bounds)
    assert torch.equal(rows, torch.cat(feats)[dev(order.astype(np.int64))])
    kept = _C.remembered_bounds(ordered)
    stacked = np.concatenate(coords)
    assert kept is None or (np.array_equal(kept[:ndim], stacked.min(0)) and np.array_equal(kept[4:4 + ndim], stacked.max(0)))


def test_collate_of_other_forms():
    """Clouds that the one call does not take: strided rows, mixed types."""
    c = [dev(random_cloud(600, 50, k)) for k in range(2)]
    f = [torch.randn(600, 2, device="cuda") for _ in c]
    want = F.collate(c, f)
    wide = [torch.stack([x, x], 2)[:, :, 0] for x in c]
    assert not wide[0].is_contiguous()
    for clouds, rows in ((wide, f), (c, [torch.stack([x, x], 2)[:, :, 0] for x in f])):
        assert all(torch.equal(a, b) for a, b in zip(F.collate(clouds, rows), want))
    mixed = F.collate([c[0].long(), c[1]], f)
    assert mixed[0].dtype == torch.int64 and torch.equal(mixed[0].int(), want[0]) and torch.equal(mixed[2], want[2])


def test_pools_beyond_values():
    """Tangents, batched features and shapes outside the library call's give what
    the tensor expressions give."""
    from torch.autograd import forward_ad
    c = torch.zeros(900, 3, dtype=torch.int32, device="cuda")
    dims = torch.tensor([0, 400, 900], dtype=torch.int32, device="cuda")
    f = torch.randn(900, 8, device="cuda")

    def mean(features, d=dims):
        return F.global_avg_pool(SparseTensor(features, c, batch_dims=d))

    with forward_ad.dual_level():
        tangent = forward_ad.unpack_dual(mean(forward_ad.make_dual(f, 2 * f))).tangent
    torch.testing.assert_close(tangent, 2 * mean(f))
    one = lambda features: mean(features, None)
    torch.testing.assert_close(torch.func.jvp(one, (f,), (3 * f,))[1], 3 * one(f))
    torch.testing.assert_close(torch.vmap(one)(torch.stack([f, -f])), torch.stack([one(f), -one(f)]))
    torch.testing.assert_close(mean(f, dims.cpu()), mean(f))
    with torch.no_grad():
        many = torch.arange(70002, device="cuda").clamp(max=900)            # 70 001 clouds, most of them empty
        total = F.global_sum_pool(SparseTensor(f, c, batch_dims=many))
        assert torch.equal(total[:900], f) and not total[900:].any()
        wide = torch.randn(3, 70000, device="cuda")
        torch.testing.assert_close(F.global_sum_pool(SparseTensor(wide, c[:3])), wide.sum(0))


def test_collate_carries_tangents():
    from torch.autograd import forward_ad
    coords = [dev(sorted_unique(random_cloud(50, 30, k))[0]) for k in range(2)]
    feats = [torch.randn(c.shape[0], 4, device="cuda") for c in coords]
    plain = F.collate(coords, feats)[2]
    with forward_ad.dual_level():
        rows = F.collate(coords, [forward_ad.make_dual(f, 2 * f) for f in feats])[2]
        assert torch.equal(forward_ad.unpack_dual(rows).tangent, 2 * plain)


@pytest.mark.parametrize("bounds", [[0, 400, 5000], [0, 900, 900], [700, 200, 900], [0, 2000, 3000]])
@pytest.mark.parametrize("rows", [900, 90000])
def test_pools_stay_inside_the_features(bounds, rows):
    """Boundaries past the last row or the wrong way round: what slices give."""
    bounds = [b * rows // 900 for b in bounds]
    f = torch.randn(rows, 64, device="cuda")
    c = torch.zeros(rows, 3, dtype=torch.int32, device="cuda")
    x = SparseTensor(f, c, batch_dims=torch.tensor(bounds, dtype=torch.int32, device="cuda"))
    parts = [f[a:b].double() for a, b in zip(bounds, bounds[1:])]
    torch.testing.assert_close(F.global_sum_pool(x).double(), torch.stack([p.sum(0) for p in parts]), rtol=1e-5, atol=1e-3)
    torch.testing.assert_close(F.global_avg_pool(x).double(), torch.stack([p.mean(0) for p in parts]), rtol=1e-5, atol=1e-5,
                               equal_nan=True)

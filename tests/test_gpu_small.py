"""Clouds around one workgroup: the sort in one launch and the split look-up of the chain."""
import numpy as np
import pytest
import torch

import c_oracle
import minuet_oracle as orc
from helpers import dev, host, random_cloud, sorted_unique
from minuet_amd.nn import functional as F
from minuet_amd.nn.functional import _C

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 1023, 1025, 4095, 4096, 4097])
@pytest.mark.parametrize("shape", ["spread", "equal rows", "one column", "wide", "batched"])
def test_sort_around_one_workgroup(n, shape):
    rng = np.random.default_rng(n)
    bd = None
    if shape == "spread":
        c = random_cloud(n, 200, n, lo=-100)
    elif shape == "equal rows":                     # far more equal keys than a part takes
        c = np.repeat(random_cloud(2, 5, n), n, axis=0)[rng.permutation(2 * n)[:n]]
    elif shape == "one column":                     # the top bits agree
        c = random_cloud(n, 3, n)
        c[:, 2] = rng.integers(-3000, 3000, size=n)
        c[0] = (1 << 20, 0, 0)
    elif shape == "wide":                           # no room for the row index beside the key
        c = rng.integers(-2 ** 20, 2 ** 20, size=(n, 3)).astype(np.int64)
    else:
        c = random_cloud(n, 30, n)
        bd = np.concatenate([[0], np.sort(rng.integers(0, n + 1, size=4)), [n]]).astype(np.int64)
    index, rows, bounds = _C.sort_coordinates(dev(c), dev(bd), return_bounds=True)
    order = orc.arg_sort_coordinates(c, bd)
    np.testing.assert_array_equal(host(index).astype(np.int64), order)
    np.testing.assert_array_equal(host(rows), c[order])
    np.testing.assert_array_equal(bounds[:3], c.min(0))
    np.testing.assert_array_equal(bounds[4:7], c.max(0))


@pytest.mark.parametrize("n", [1, 5, 511, 513, 2039, 4096, 4500])
@pytest.mark.parametrize("kernel,extent,halves", [(3, 16, True), (3, 400, True), (2, 16, False)])
def test_map_lists_of_small_clouds(n, kernel, extent, halves):
    c, _ = sorted_unique(random_cloud(n, extent, n + kernel, lo=-extent // 2))
    c = c[np.random.default_rng(n).permutation(c.shape[0])]
    check_map_lists(c, orc.generate_kernel_offsets(3, kernel, 1, 1))


def look_up(rows, off):
    """The map by a table of the rows (the C oracle packs a row into one key)."""
    at = {row: i for i, row in enumerate(map(tuple, rows.tolist()))}
    return np.array([[at.get(row, -1) for row in map(tuple, (rows + step).tolist())] for step in off], dtype=np.int32)


def check_map_lists(c, off, query=None):
    index, rows, built = _C.sorted_kernel_map_lists(dev(c), off.astype(np.int64))
    order = orc.arg_sort_coordinates(c)
    np.testing.assert_array_equal(host(index).astype(np.int64), order)
    np.testing.assert_array_equal(host(rows), c[order])
    ref = query(c[order], off) if query else c_oracle.query(c[order], c[order], off.astype(np.int32))
    sizes = orc.compute_kernel_map_sizes(ref)
    by_size = orc.stable_size_order(sizes)
    ein, eout, _ = orc.kernel_map_pair_lists(ref[by_size])
    np.testing.assert_array_equal(built["sizes_host"], np.asarray(sizes)[by_size])
    np.testing.assert_array_equal(host(built["in_idx"]), ein)
    np.testing.assert_array_equal(host(built["out_idx"]), eout)


# clouds that the one launch turns down: more rows than a part takes agree in the top bits of the key, and keys
# that leave no room for the row index (59 bits, which the chain's query takes, and 66, which it does not)
@pytest.mark.parametrize("n", [500, 4000])
@pytest.mark.parametrize("shape", ["crowded", "wide", "too wide"])
@pytest.mark.parametrize("kernel", [3, 4, 5])
def test_map_lists_of_clouds_turned_down(n, shape, kernel):
    if shape == "crowded":
        c = random_cloud(3 * n, 3, n + kernel)
        c[:, 2] = np.random.default_rng(n).integers(-3000, 3000, size=3 * n)
        c[0] = (1 << 20, 0, 0)
    else:
        c = random_cloud(2 * n, 24, n, lo=-12, dtype=np.int64)
        c[0] = (1 << 19, (1 << 18) + 3, (1 << 19) + 1) if shape == "wide" else (1 << 21, 1 << 21, 1 << 21)
    c, _ = sorted_unique(c)
    c = np.concatenate([c[:n // 2], c[-(n // 2):]])
    check_map_lists(c[np.random.default_rng(n).permutation(c.shape[0])], orc.generate_kernel_offsets(3, kernel, 1, 1), look_up)


# 125 and 49 offsets (two a lane), offsets past the cloud, coordinates of 64 bits far apart, one to four
# dimensions; workgroups that hear of the others' counts, and such that count for themselves
@pytest.mark.parametrize("patience", [None, "0"])
@pytest.mark.parametrize("n,ndim,kernel,dilation,dtype", [
    (4096, 3, 5, 1, np.int32), (2039, 3, 3, 2, np.int64), (700, 2, 7, 1, np.int32), (65, 4, 3, 1, np.int32),
    (3000, 1, 3, 1, np.int64), (1500, 3, 5, 40, np.int32), (4096, 3, 4, 1, np.int32)])
def test_map_lists_in_one_launch(n, ndim, kernel, dilation, dtype, patience, monkeypatch):
    if patience is not None:
        monkeypatch.setenv("MINUET_MAP_PATIENCE", patience)
    extent = int(round((3 * n) ** (1 / ndim)))
    c, _ = sorted_unique(random_cloud(n, extent, n + kernel, ndim=ndim, lo=-extent // 2, dtype=dtype))
    if dtype == np.int64:
        c[-1] += 1 << 40 // ndim
    c = c[np.random.default_rng(n).permutation(c.shape[0])]
    check_map_lists(c, orc.generate_kernel_offsets(ndim, kernel, 1, dilation))


# the chain of launches under 65 to 128 offsets that come in pairs (64 kept at most), with the largest that do
# and one that does not take it; one tile more than one, several buckets, windows of more than one chunk
@pytest.mark.parametrize("n,ndim,kernel,dilation,dtype", [
    (4097, 3, 5, 1, np.int32), (70000, 3, 5, 1, np.int64), (20000, 2, 11, 1, np.int32), (9000, 1, 127, 1, np.int32),
    (9000, 1, 129, 1, np.int32), (6000, 3, 5, 7, np.int32), (12000, 3, 4, 1, np.int32)])
def test_map_lists_of_many_offsets(n, ndim, kernel, dilation, dtype):
    extent = int(round((4 * n) ** (1 / ndim)))
    c, _ = sorted_unique(random_cloud(2 * n, extent, n + kernel, ndim=ndim, lo=-extent // 2, dtype=dtype))
    c = c[np.random.default_rng(n).permutation(c.shape[0])][:n]
    check_map_lists(c, orc.generate_kernel_offsets(ndim, kernel, 1, dilation))


def test_map_lists_of_equal_rows():
    """The one launch turns such a cloud down, whoever of the workgroups sees it."""
    c = random_cloud(3000, 12, 8, duplicates=0.3)
    order = orc.arg_sort_coordinates(c)
    off = orc.generate_kernel_offsets(3, 3, 1, 1)
    index, rows, built = _C.sorted_kernel_map_lists(dev(c), off.astype(np.int64))
    np.testing.assert_array_equal(host(index).astype(np.int64), order)
    whole = _C.kernel_map_build(rows, rows, off.astype(np.int64), None, None, reorder=True, want_masks=False, want_lists=True)
    for name in ("in_idx", "out_idx"):
        assert torch.equal(built[name], whole[name])
    np.testing.assert_array_equal(built["sizes_host"], whole["sizes_host"])


# The library's scratch memory begins with integers that look like the words the workgroups of the next call
# answer each other with: the call's number (1, 2, ... after a reset) above 13 bits of a count.  A sort of more than
# 4 096 rows leaves its extremes there, a batch that is collated its 64-bit coordinates.
@pytest.mark.parametrize("patience", [None, "0"])
@pytest.mark.parametrize("left_by", ["sort", "collate"])
def test_map_lists_after_calls_that_leave_such_words(left_by, patience, monkeypatch):
    if patience is not None:
        monkeypatch.setenv("MINUET_MAP_PATIENCE", patience)
    c, _ = sorted_unique(random_cloud(600, 14, 5, lo=-7))
    off = orc.generate_kernel_offsets(3, 3, 1, 1)
    for _ in range(2):
        torch.cuda.synchronize()
        _C.cuda_device_reset()
        for number in range(2, 18, 2):           # (one number for the sort or the batch, one for the map)
            rows = random_cloud(5000 if left_by == "sort" else 300, 1 << 13, number, lo=number << 13, dtype=np.int64)
            if left_by == "sort":
                _C.sort_coordinates(dev(rows), None)
            else:
                F.collate([dev(rows)])
            check_map_lists(c, off)

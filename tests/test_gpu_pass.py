"""The build of a whole pass (levels and maps at once) against the single calls."""
import ctypes

import numpy as np
import pytest
import torch

import minuet_amd as minuet
from helpers import dev, random_cloud, sorted_unique
from minuet_amd.nn.functional import _C
from minuet_amd.nn.passplan import PassPlan
from minuet_amd.unet import SparseUNet
from minuet_amd.utils.helpers import generate_kernel_offsets

pytestmark = pytest.mark.gpu


def offsets_of(source_stride, kernel_size, dilation):
    return np.ascontiguousarray(generate_kernel_offsets(3, kernel_size, source_stride, dilation), dtype=np.int64)


@pytest.mark.parametrize("n,extent,stride,batches,ctype,itype", [
    (1, 5, 2, 1, np.int32, None), (70, 9, 2, 1, np.int32, None), (5000, 40, 2, 3, np.int32, np.int32),
    (5000, 40, 3, 2, np.int64, np.int64), (30000, 500, 2, 4, np.int32, np.int64), (200, 6, 4, 7, np.int32, np.int32)])
def test_pass_build_equals_single_calls(n, extent, stride, batches, ctype, itype):
    rng = np.random.default_rng(n)
    bd = None
    if batches > 1:
        cuts = np.sort(rng.integers(0, n, size=batches - 1))
        bd = np.concatenate([[0], cuts, [n]]).astype(itype)
    c, bd = sorted_unique(random_cloud(n, extent, n, lo=-extent // 2, dtype=ctype), bd)
    s1, s2, s4 = (1,) * 3, (stride,) * 3, (stride * stride,) * 3
    one = (1, 1, 1)
    sub = [(s, s, (3, 3, 3), one) for s in (s1, s2, s4)]
    down = [(s1, s2, (2, 2, 2), one), (s2, s4, (2, 2, 2), one), (s2, s4, (3, 3, 3), one)]
    requests = [("coords", s1, s2), ("coords", s2, s4)]
    for key in sub:
        requests += [("dense", key), ("groups", key), ("tables", key, True)]
    for key in down:
        requests += [("dense", key), ("invert", key), ("tables", key, False)]
    index_dtype = torch.int32 if ctype == np.int32 else torch.int64
    if itype is not None:
        index_dtype = torch.int32 if itype == np.int32 else torch.int64
    plan = PassPlan(requests, offsets_of, s1, index_dtype)
    coords, dims = dev(c), dev(bd)
    for _ in range(2):                                   # the second build finds the bitmaps the first has cleared
        built = plan.build(coords, dims, None)
    levels = {s1: (coords, dims)}
    for source, target in ((s1, s2), (s2, s4)):
        levels[target] = _C.target_coordinates(*levels[source], target)
        got = built.coordinates[target]
        assert torch.equal(got[0], levels[target][0]) and got[1] == target
        assert (dims is None and got[2] is None) or torch.equal(got[2], levels[target][1])
    for key in sub + down:
        source, target, kernel, dilation = key
        offsets = offsets_of(source, kernel, dilation)
        dense, _ = _C.kernel_map_dense(levels[source][0], levels[target][0], offsets, levels[source][1],
                                       levels[target][1])
        assert torch.equal(built.dense(key, built.coordinates[source][0]), dense), key
        assert built.dense(key, built.coordinates[source][0].clone()) is None       # another tensor: not served
        num_sources = levels[source][0].shape[0]
        if key in down:
            assert torch.equal(built.inverse(key), _C.kernel_map_invert(dense, num_sources)), key
        else:
            ref = _C.kernel_map_offset_groups(dense, offsets)
            got = built.groups(key, built.coordinates[source][0])
            rows = ref.head[1:10].tolist()
            assert torch.equal(got.head[:10], ref.head[:10]) and torch.equal(got.rank, ref.rank)
            for j, count in enumerate(rows):
                lo = j * dense.shape[1]
                assert torch.equal(got.src[lo:lo + count, :3], ref.src[lo:lo + count, :3])
        if index_dtype == torch.int32:
            reorder = key in sub
            ref = _C.kernel_map_tables(dense, num_sources, reorder)
            got = built.tables(key, built.coordinates[source][0], reorder)
            assert np.array_equal(got.sizes_host, ref["sizes_host"])
            for name in ("source_masks", "target_masks", "in_idx", "out_idx"):
                assert torch.equal(getattr(got, name), ref[name]), (key, name)
            assert torch.equal(got.kernel_map_sizes, ref["sizes"])
            if reorder:
                assert np.array_equal(got.order_host, ref["order_host"])
                assert torch.equal(got.kernel_map_order, ref["order"])


@pytest.mark.parametrize("kind", ["fp16", "fp32"])
def test_second_pass_of_a_network_equals_its_first(kind):
    """The second pass after a reset builds everything at once; other clouds, the
    same cloud again and a cache left alone give what a fresh cache gives."""
    dtype = torch.float16 if kind == "fp16" else torch.float32
    torch.manual_seed(0)
    net = SparseUNet(4, 16, dtype=dtype, device="cuda").eval()
    cache = minuet.nn.KernelMapCache(3, torch.int32, "cuda")
    with torch.no_grad():
        for seed, n in ((1, 3000), (2, 4100), (1, 3000), (3, 900)):
            c, bd = sorted_unique(random_cloud(n, 30, seed, lo=-9), np.array([0, n // 3, n], dtype=np.int32))
            x = minuet.SparseTensor(torch.randn(c.shape[0], 4, device="cuda").to(dtype), dev(c), batch_dims=dev(bd))
            cache.reset()
            minuet.set_kernel_map_cache(net, cache)
            y = net(x)
            assert (cache._built is not None) == (seed != 1 or cache._pass_plan is not None)
            again = net(x)                                       # maps kept
            minuet.set_kernel_map_cache(net, minuet.nn.KernelMapCache(3, torch.int32, "cuda"))
            ref = net(x)
            assert torch.equal(y.C, ref.C) and torch.equal(y.F, ref.F) and torch.equal(again.F, ref.F)
            assert torch.equal(y.batch_dims, ref.batch_dims)
    assert cache.num_coordinate_builds == 16 and cache.num_map_builds == 36


def test_build_belongs_to_the_levels_before_it():
    """Threads that take turns on one stream: what another pass has left there in
    between is not built into this one's block, and the other goes on."""
    one, two = (1, 1, 1), (2, 2, 2)
    requests = [("coords", one, two), ("dense", (one, one, (3, 3, 3), one)), ("dense", (one, two, (2, 2, 2), one))]
    clouds = [dev(sorted_unique(random_cloud(n, 40, n))[0]) for n in (300, 5000)]
    plans = [PassPlan(requests, offsets_of, one, torch.int32) for _ in clouds]
    sizes = [_C.pass_levels(c, None, None, p.levels, p.num_levels, p.maps)[0] for c, p in zip(clouds, plans)]
    stores = [torch.empty(size, dtype=torch.uint8, device="cuda") for size in sizes]
    with pytest.raises(RuntimeError, match="another cloud or other lists"):
        _C.pass_build(clouds[0], None, plans[0].levels, plans[0].maps, stores[0])
    _C.pass_build(clouds[1], None, plans[1].levels, plans[1].maps, stores[1])
    dense, _ = _C.kernel_map_dense(clouds[1], clouds[1], offsets_of(one, (3, 3, 3), one), None, None)
    at = plans[1].maps[plans[1].map_of[requests[1][1]]].at[0]
    assert torch.equal(stores[1].view(torch.int32)[at // 4:at // 4 + dense.numel()].view_as(dense), dense)
    assert plans[0].build(clouds[0], None, None) is not None

    # a count of target coordinates and the levels of a pass share their block
    lib, stride, count = _C.load_library(), (ctypes.c_int64 * 3)(2, 2, 2), ctypes.c_int64(0)
    stream = _C._stream(clouds[0].device)
    _C._check(lib.mnt_target_coordinates_count(clouds[0].data_ptr(), clouds[0].shape[0], 3, 0, stride, None, 1, 0, None,
                                               ctypes.byref(count), stream))
    assert _C.pass_levels(clouds[1], None, None, plans[1].levels, plans[1].num_levels, plans[1].maps)
    out = torch.empty(count.value, 3, dtype=torch.int32, device="cuda")
    assert lib.mnt_target_coordinates_fill(out.data_ptr(), None, stream) != 0
    _C.pass_build(clouds[1], None, plans[1].levels, plans[1].maps, stores[1])


def test_tables_wait_for_their_own_flag():
    """The word in pinned memory that says a map's tables are complete may hold the
    order of an earlier map there, whose first two entries then read as a number:
    whichever number the pass waits for, it is not taken for the flag."""
    one, key = (1, 1, 1), ((1, 1, 1), (1, 1, 1), (3, 3, 3), (1, 1, 1))
    offsets = offsets_of(one, (3, 3, 3), one)
    cloud = dev(sorted_unique(random_cloud(60000, 300, 5))[0])
    dense, _ = _C.kernel_map_dense(cloud, cloud, offsets, None, None)
    expected = _C.kernel_map_tables(dense, cloud.shape[0], True)
    plan = PassPlan([("dense", key), ("tables", key, True)], offsets_of, one, torch.int32)
    for number in range(1, 27):
        # a map whose order starts (number, 0): fewest hits under that offset, then under the first
        counts = np.full(27, 40)
        counts[[0, number]] = 20, 10
        earlier = torch.full((27, 64), -1, dtype=torch.int32)
        for o, count in enumerate(counts):
            earlier[o, :count] = torch.arange(count, dtype=torch.int32)
        torch.cuda.synchronize()
        _C.cuda_device_reset()                           # the numbers start again
        order = _C.kernel_map_tables(earlier.cuda(), 64, True)["order_host"]
        assert order[0] == number and order[1] == 0
        built = plan.build(cloud, None, np.array([0, 0, 0, 0, 299, 299, 299, 0], dtype=np.int64))
        got = built.tables(key, cloud, True)
        assert np.array_equal(got.sizes_host, expected["sizes_host"])
        assert np.array_equal(got.order_host, expected["order_host"])


def test_transposed_layer_changes_its_dataflow_in_a_planned_pass():
    """Its tables are not on the pass's list, and the layer before it, which shares
    the map, ran past Python: they come from the map that was built."""
    gen = torch.Generator().manual_seed(1)
    coordinates = torch.unique(torch.randint(0, 24, (5000, 3), generator=gen, dtype=torch.int32), dim=0).cuda()
    coordinates = coordinates[minuet.nn.functional.build_sorted_index(coordinates)]
    down = minuet.nn.SparseConv3d(32, 64, 2, stride=2, dtype=torch.float16, device="cuda")
    up = minuet.nn.SparseConv(3, 64, 32, 2, stride=2, transposed=True, dtype=torch.float16, device="cuda")
    net = torch.nn.Sequential(down, up)
    cache = minuet.nn.KernelMapCache(ndim=3, dtype=torch.int32, device="cuda")
    minuet.set_kernel_map_cache(net, cache)
    x = minuet.SparseTensor(torch.randn(len(coordinates), 32, generator=gen).half().cuda(), coordinates)
    with torch.no_grad():
        for _ in range(3):
            first = net(x).F
            cache.reset()
        up.tunable_config["dataflow"] = "gather_gemm_scatter"
        other = net(x).F
    assert torch.allclose(first, other, rtol=4e-3, atol=4e-3)


@pytest.mark.parametrize("size", [(96, 64, 64), (7, 130, 66)])
def test_levels_of_a_full_block(size):
    """Tiles of the levels' bitmaps with more rows than their keys fit in LDS
    together, and words of which some rows do: asked for one by one, then planned."""
    grids = torch.meshgrid(*(torch.arange(n, dtype=torch.int32) for n in size), indexing="ij")
    coordinates = torch.stack([g.flatten() for g in grids], 1).cuda()
    keep = torch.rand(len(coordinates), generator=torch.Generator().manual_seed(1)) > 0.02
    coordinates = coordinates[keep.cuda()].contiguous()
    net = torch.nn.Sequential(minuet.nn.SparseConv3d(8, 8, 2, stride=2, dtype=torch.float16, device="cuda"),
                              minuet.nn.SparseConv3d(8, 8, 2, stride=2, dtype=torch.float16, device="cuda"))
    cache = minuet.nn.KernelMapCache(ndim=3, dtype=torch.int32, device="cuda")
    minuet.set_kernel_map_cache(net, cache)
    x = minuet.SparseTensor(torch.ones(len(coordinates), 8, device="cuda").half(), coordinates)
    expected = torch.unique(torch.div(coordinates, 4, rounding_mode="floor") * 4, dim=0)
    with torch.no_grad():
        for _ in range(3):
            out = net(x)
            assert out.C.equal(expected)
            assert net[0](x).C.equal(torch.unique(torch.div(coordinates, 2, rounding_mode="floor") * 2, dim=0))
            cache.reset()


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_a_planned_pass_without_tiles_asks_nothing_about_them(dtype, monkeypatch):
    """Neither which stream is current nor what tiles would have saved: each is a
    microsecond or more of a layer that takes thirty with its map."""
    c, _ = sorted_unique(random_cloud(3000, 20, 5, lo=-9), None)
    conv = minuet.nn.SparseConv3d(32, 32, 3, dtype=dtype, device="cuda")
    cache = minuet.nn.KernelMapCache(3, torch.int32, "cuda")
    conv.set_kernel_map_cache(cache)
    x = minuet.SparseTensor(torch.randn(c.shape[0], 32, device="cuda").to(dtype), dev(c))
    with torch.no_grad():
        first = conv(x).F
        for _ in range(2):
            cache.reset()
            assert torch.equal(conv(x).F, first)
        calls = []
        monkeypatch.setattr(torch.cuda, "current_stream", lambda *a: calls.append("stream"))
        monkeypatch.setattr(type(cache), "_note_tiles", lambda *a: calls.append("tiles"))
        cache.reset()
        assert torch.equal(conv(x).F, first) and cache._built is not None
        cache.reset()
        assert not calls

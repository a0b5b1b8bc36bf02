"""Host-side API behaviour that needs no GPU: SparseTensor validation, helper
functions, module construction, tunable-config round trips, the drop-in alias."""
import json

import numpy as np
import pytest
import torch

import minuet_amd as minuet
from minuet_amd.utils.helpers import as_tuple


def test_alias_package_points_at_the_same_objects():
    import minuet as alias
    import minuet.nn.functional as AF
    from minuet.nn import SparseConv3d, KernelMapCache
    from minuet.utils.helpers import generate_kernel_offsets
    assert alias.SparseTensor is minuet.SparseTensor
    assert SparseConv3d is minuet.nn.SparseConv3d and KernelMapCache is minuet.nn.KernelMapCache
    assert AF.sparse_convolution_forward is minuet.nn.functional.sparse_convolution_forward
    assert generate_kernel_offsets is minuet.utils.helpers.generate_kernel_offsets
    for name in ("set_kernel_map_cache", "autotune", "load_tunable_config", "dump_tunable_config",
                 "set_gemm_parallel_level"):
        assert getattr(alias, name) is getattr(minuet, name)
    for name in ("arg_sort_coordinates", "build_sorted_index", "query_sorted_index_with_offsets",
                 "unique_coordinates", "compute_kernel_map_masks", "compute_kernel_map_sizes",
                 "cuda_time_gather", "cuda_time_scatter", "cuda_time_gemm", "sparse_convolution_forward",
                 "set_gemm_parallel_level", "cuda_buffer_total_size", "cuda_buffer_used_size",
                 "cuda_free_buffers", "cuda_set_buffer_growth", "cuda_set_buffer_page_size",
                 "cuda_preallocate_buffer", "cuda_reset_error", "global_avg_pool", "global_max_pool",
                 "global_sum_pool", "cat"):
        assert hasattr(AF, name), name


def test_as_tuple():
    assert as_tuple(2) == (2, 2, 2)
    assert as_tuple((1, 2), size=2) == (1, 2)
    assert as_tuple([3, 4, 5]) == (3, 4, 5)
    with pytest.raises(ValueError, match="kernel_size must be a scalar or a iterable of size 3"):
        as_tuple((1, 2), size=3, name="kernel_size")


def test_sparse_tensor_validation_and_properties():
    f = torch.randn(5, 4)
    c = torch.zeros((5, 3), dtype=torch.int32)
    x = minuet.SparseTensor(f, c, stride=2, batch_dims=torch.tensor([0, 2, 5]))
    assert x.stride == (2, 2, 2) and x.batch_size == 2 and x.n == 5 and x.ndim == 3
    assert x.num_features == 4 and x.shape == (5, 4) and x.dtype == torch.float32
    assert minuet.SparseTensor(f, c, batch_dims=torch.tensor([0, 5])).batch_dims is None
    assert minuet.SparseTensor(f, c).batch_size == 1
    with pytest.raises(ValueError, match="must be a 2-D tensor"):
        minuet.SparseTensor(f, c[:, 0])
    with pytest.raises(ValueError, match="features tensor indicate 5 coordinates but expected 4"):
        minuet.SparseTensor(f, c[:4])
    with pytest.raises(ValueError, match="must be int32 or int64"):
        minuet.SparseTensor(f, c.float())
    with pytest.raises(ValueError, match="strides must be a scalar"):
        minuet.SparseTensor(f, c, stride=(1, 2))
    with pytest.raises(ValueError, match="different from expected"):
        x.F = torch.randn(4, 4)
    x.F = torch.ones(5, 4)
    assert x.half().dtype == torch.float16 and x.half().C is x.C
    y = x.clone()
    assert y.C is not x.C and torch.equal(y.C, x.C) and torch.equal(y.batch_dims, x.batch_dims)
    z = x.to(dtype=torch.float64, copy=True)
    assert z.dtype == torch.float64 and z.C.dtype == torch.int32 and x.dtype == torch.float32
    assert x.detach().F.requires_grad is False
    assert x.contiguous() is x and x.cpu() is x


def test_conv_module_construction():
    conv = minuet.nn.SparseConv3d(8, 16, 3, bias=True)
    assert conv.kernel.shape == (27, 8, 16) and conv.bias.shape == (16,)
    bound = 1.0 / np.sqrt(8 * 27)
    assert conv.kernel.abs().max() <= bound and conv.bias.abs().max() <= bound
    assert conv.tunable_config == {"threshold": -1, "gather_tile_size": 0, "scatter_tile_size": 0,
                                   "dataflow": "auto"}
    assert repr(conv) == "SparseConv3d(8, 16, kernel_size=(3, 3, 3))"
    up = minuet.nn.SparseConv(3, 8, 4, 2, stride=2, transposed=True)
    assert "stride=(2, 2, 2)" in repr(up) and "transposed=True" in repr(up) and "bias=False" in repr(up)
    assert up.kernel.abs().max() <= 1.0 / np.sqrt(4 * 8)          # transposed: fan = out_channels
    assert minuet.nn.SparseConv3d(4, 4, 1).is_trivial and not conv.is_trivial
    assert set(conv.state_dict()) == {"kernel", "bias"}
    d = minuet.nn.SparseConv3d(4, 4, 3, dilation=2)
    assert "dilation=(2, 2, 2)" in repr(d)
    cache = minuet.nn.KernelMapCache(ndim=3, dtype=torch.int32, device="cpu")
    for m in (conv, d, minuet.nn.SparseConv3d(4, 4, 3, stride=2)):
        m.set_kernel_map_cache(cache)
    assert conv._allow_shortcut_matmul and not d._allow_shortcut_matmul
    x = minuet.SparseTensor(torch.randn(3, 8), torch.zeros((3, 3), dtype=torch.int32))
    with pytest.raises(ValueError, match="Kernel map cache must be specified"):
        minuet.nn.SparseConv3d(8, 8, 3)(x)


def test_trivial_conv_and_wrappers_on_cpu():
    x = minuet.SparseTensor(torch.randn(6, 4), torch.arange(18, dtype=torch.int32).view(6, 3),
                            batch_dims=torch.tensor([0, 2, 6]))
    conv = minuet.nn.SparseConv3d(4, 5, 1, bias=True)
    with torch.no_grad():
        y = conv(x)
    torch.testing.assert_close(y.F, x.F @ conv.kernel[0] + conv.bias)
    assert y.C is x.C and y.batch_dims is x.batch_dims
    r = minuet.nn.ReLU()(x)
    assert (r.F >= 0).all() and r.C is x.C
    assert minuet.nn.LeakyReLU(0.1)(x).F.shape == x.F.shape and minuet.nn.ReLU6()(x).F.max() <= 6
    bn = minuet.nn.BatchNorm(4).eval()
    torch.testing.assert_close(bn(x).F, x.F / np.sqrt(1 + 1e-5), rtol=1e-5, atol=1e-6)
    both = minuet.nn.functional.cat([x, r])
    assert both.F.shape == (6, 8) and both.C is x.C
    avg = minuet.nn.GlobalAvgPool()(x)
    torch.testing.assert_close(avg, torch.stack([x.F[:2].mean(0), x.F[2:].mean(0)]))
    torch.testing.assert_close(minuet.nn.GlobalSumPool()(x)[1], x.F[2:].sum(0))
    torch.testing.assert_close(minuet.nn.GlobalMaxPool()(x)[0], x.F[:2].max(0)[0])
    single = minuet.SparseTensor(x.F, x.C)
    torch.testing.assert_close(minuet.nn.GlobalAvgPool()(single), x.F.mean(0))


def test_tunable_config_round_trip(tmp_path):
    net = torch.nn.Sequential(minuet.nn.SparseConv3d(4, 8, 3), minuet.nn.ReLU(),
                              torch.nn.Sequential(minuet.nn.SparseConv3d(8, 8, 3)))
    cfg = minuet.dump_tunable_config(net)
    assert set(cfg) == {"0", "1", "2"} and cfg["1"] == {} and set(cfg["2"]) == {"0"}
    cfg = json.loads(json.dumps(cfg))
    cfg["0"]["threshold"] = 0.25
    cfg["2"]["0"]["gather_tile_size"] = 4
    other = torch.nn.Sequential(minuet.nn.SparseConv3d(4, 8, 3), minuet.nn.ReLU(),
                                torch.nn.Sequential(minuet.nn.SparseConv3d(8, 8, 3)))
    minuet.load_tunable_config(other, cfg)
    assert other[0].tunable_config["threshold"] == 0.25
    assert other[2][0].tunable_config["gather_tile_size"] == 4
    path = tmp_path / "cfg.json"
    path.write_text(json.dumps(cfg))
    again = torch.nn.Sequential(minuet.nn.SparseConv3d(4, 8, 3), minuet.nn.ReLU(),
                                torch.nn.Sequential(minuet.nn.SparseConv3d(8, 8, 3)))
    minuet.autotune(again, None, [], cache_path=str(path))        # existing file: load, never run
    assert again[0].tunable_config["threshold"] == 0.25


def test_set_kernel_map_cache_is_recursive():
    cache = minuet.nn.KernelMapCache(ndim=3, dtype=torch.int32, device="cpu")
    net = torch.nn.Sequential(minuet.nn.SparseConv3d(4, 8, 3),
                              torch.nn.Sequential(minuet.nn.ReLU(), minuet.nn.SparseConv3d(8, 8, 3)))
    assert minuet.set_kernel_map_cache(net, cache) is net
    assert net[0]._kernel_map_cache is cache and net[1][1]._kernel_map_cache is cache


def test_random_unique_points():
    from minuet_amd.utils.random import random_unique_points
    pts = random_unique_points(3, 200, -2, 4)
    assert pts.shape == (200, 3) and pts.min() >= -2 and pts.max() <= 4
    assert len({tuple(p) for p in pts.tolist()}) == 200
    with pytest.raises(ValueError):
        random_unique_points(2, 10, 0, 2)
    assert len({tuple(p) for p in random_unique_points(2, 9, 0, 2).tolist()}) == 9


def test_auto_dataflow_rule():
    """Which layer shapes ``dataflow="auto"`` sends to the single-kernel form:
    16-bit rows of up to 128 bytes with up to 128 output channels, rows of up
    to 256 bytes with up to 64 output channels under kernels of more than 8
    offsets, and small fp32 layers with 2^D kernels."""
    prefers = minuet.nn.functional.prefers_implicit
    half, single = torch.float16, torch.float32
    assert prefers(27, 32, 32, half) and prefers(27, 64, 128, half) and prefers(8, 64, 128, torch.bfloat16)
    assert not prefers(27, 64, 256, half)                 # too many output channels
    assert prefers(27, 32, 256, half) and prefers(8, 8, 132, half) and prefers(125, 16, 512, half)      # short rows
    assert not prefers(64, 32, 256, half) and not prefers(216, 32, 160, half) and not prefers(27, 40, 160, half)
    assert prefers(27, 128, 64, half) and not prefers(27, 128, 128, half)
    assert not prefers(8, 128, 64, half)                  # strided 2^3 kernel: one hit in eight
    assert not prefers(27, 256, 64, half)                 # 512-byte rows
    assert not prefers(27, 30, 32, half)                  # rows not a multiple of 16 bytes
    assert prefers(8, 32, 32, single) and not prefers(27, 32, 32, single) and not prefers(8, 64, 64, single)


def test_fp32_rule_stops_at_the_rows_that_can_be_addressed():
    """Narrow layers go to the single-kernel form at any size but one: features
    of 4 GiB, which that form cannot address, stay with the three kernels."""
    prefers, single = minuet.nn.functional.prefers_hits, torch.float32
    most = (0xFFFFF000 - 1) // (32 * 4)
    for offsets in (8, 27):
        assert prefers(offsets, 32, 32, single, most) and not prefers(offsets, 32, 32, single, most + 1)
    assert not prefers(27, 4, 4, single, 2 ** 28) and prefers(27, 4, 4, single, 2 ** 27)


def test_fp32_rule_follows_the_kernel_size():
    """Wider layers change over at fewer rows the more offsets they have."""
    prefers, single = minuet.nn.functional.prefers_hits, torch.float32
    assert prefers(8, 64, 128, single, 13000) and not prefers(8, 64, 128, single, 14000)
    assert prefers(27, 64, 64, single, 18900) and not prefers(27, 64, 64, single, 19100)
    assert prefers(125, 64, 64, single, 4000) and not prefers(125, 64, 64, single, 4200)
    assert prefers(125, 32, 32, single, 100000)


def test_fp32_rule_for_few_input_channels():
    """Past the line product rows outgrow the caches: few input channels never leave the single-kernel form, a
    few more come back to it."""
    prefers, single = minuet.nn.functional.prefers_hits, torch.float32
    assert all(prefers(27, 16, 256, single, rows) for rows in (1000, 50000, 10 ** 6))
    for offsets, back in ((27, 250000), (125, 130000)):
        assert prefers(offsets, 48, 64, single, 1000) and prefers(offsets, 48, 64, single, back)
        assert not prefers(offsets, 48, 64, single, 30000) and not prefers(offsets, 48, 64, single, back - 1)
        assert not prefers(offsets, 64, 64, single, 10 ** 6)
    assert not prefers(8, 48, 64, single, 10 ** 6)
    most = (0xFFFFF000 - 1) // (48 * 4)
    assert prefers(27, 48, 64, single, most) and not prefers(27, 48, 64, single, most + 1)


# (channels, rows) where cutting the channels was measured slower than one offset, and where faster
@pytest.mark.parametrize("cin, cout, slower, faster", [
    (64, 32, 60000, 30000), (96, 64, 30000, 8000), (48, 128, 20000, 4500), (80, 48, 30000, 20000), (96, 128, 20000, 9000),
    (256, 32, None, 9000), (160, 128, None, 9000), (48, 256, None, 9000)])
def test_pointwise_layers_are_cut_where_that_is_faster(cin, cout, slower, faster):
    most = minuet.nn.functional.pieces_rows_limit(cin, cout, torch.float32)
    assert faster <= most and (slower is None or most < slower)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_rows_that_the_single_kernel_form_addresses(dtype):
    limit = minuet.nn.functional.implicit_rows_limit
    for channels in (4, 100, 128, 256):
        most = limit(channels, dtype)
        row = channels * dtype.itemsize
        assert most * row < 0xFFFFF000 <= (most + 1) * row      # (what the library refuses)


def test_lookahead_layout_places_every_output():
    """The plan of a look-ahead session (no GPU needed): every output of every
    recipe entry gets a 256-byte aligned place of its own inside one allocation,
    entries that need a level or map nobody builds are refused."""
    import torch
    from minuet_amd.nn.functional import _C
    from minuet_amd.nn.lookahead import AheadLayout
    cache = minuet.nn.KernelMapCache(ndim=3, dtype=torch.int32, device="cpu")
    one, two = (1, 1, 1), (2, 2, 2)
    sub = (one, one, (3, 3, 3), one)
    down = (one, two, (2, 2, 2), one)
    recipe = (("dense", sub), ("coords", one, two), ("dense", down), ("tables", down, True), ("invert", down))
    layout = AheadLayout(recipe, cache._kernel_offsets, one, 1 << 14, 3, torch.int32, torch.int32, 2)
    assert layout.num_levels == 2 and len(layout.items) == 5
    assert [item.kind for item in layout.items] == [_C.AHEAD_DENSE, _C.AHEAD_COORDS, _C.AHEAD_DENSE,
                                                    _C.AHEAD_TABLES, _C.AHEAD_INVERT]
    assert layout.items[3].dense_item == 2 and layout.items[4].dense_item == 2 and layout.items[3].reorder == 1
    assert layout.items[0].num_offsets == 27 and layout.items[2].num_offsets == 8
    spans = []
    for places, (_, _, _, sizes) in zip(layout.places, layout.plan):
        for place, size in zip(places, sizes):
            if size:
                assert place % 256 == 0
                spans.append((place, place + size))
    spans.sort()
    assert all(a[1] <= b[0] for a, b in zip(spans, spans[1:])) and spans[-1][1] <= layout.total
    layout.bind(1 << 20)
    assert layout.items[0].out0 == (1 << 20) + layout.places[0][0]
    assert layout.items[1].out1 == (1 << 20) + layout.places[1][1]          # batch boundaries of the new level
    for bad in ((("tables", sub, True),), (("coords", two, (4, 4, 4)),), (("dense", down),), ()):
        with pytest.raises(ValueError):
            AheadLayout(bad, cache._kernel_offsets, one, 1 << 14, 3, torch.int32, None, 1)


def test_padded_weights_are_those_of_the_present_kernel(monkeypatch):
    """A kernel put in another's place is packed anew, also where the allocator
    hands it the same memory."""
    monkeypatch.setattr(minuet.nn.functional, "pack_weights", lambda weights: weights.clone())
    conv = minuet.nn.SparseConv3d(3, 8, 3)
    with torch.no_grad():
        for value in range(1, 40):
            del conv.kernel
            conv.kernel = torch.nn.Parameter(torch.full((27, 3, 8), float(value)))
            weights, packed = conv._packed_kernel(1)
            assert bool((weights[:, :3] == value).all()) and bool((packed[:, :3] == value).all())


def test_what_a_library_call_may_stand_in_for():
    """Pools and collating are one library call only where nothing but values counts."""
    from torch.autograd import forward_ad
    from torch.utils._python_dispatch import TorchDispatchMode
    from minuet_amd.nn.functional import _C
    x, seen = torch.ones(4, 3), []
    assert _C.plain([x, x]) and not _C.plain([x, torch.ones(2, requires_grad=True)])
    with torch.no_grad():
        assert _C.plain([torch.ones(2, requires_grad=True)])
    with forward_ad.dual_level():
        assert not _C.plain([x, forward_ad.make_dual(x, x)]) and _C.plain([x])
    torch.vmap(lambda t: seen.append(_C.plain([t])) or t)(x)
    torch.func.jvp(lambda t: seen.append(_C.plain([t])) or t, (x,), (x,))
    torch.func.grad(lambda t: seen.append(_C.plain([t])) or t.sum())(x)
    torch.jit.trace(lambda t: seen.append(_C.plain([t])) or t + 1, x, check_trace=False)
    with TorchDispatchMode():
        seen.append(_C.plain([x]))
    assert seen and not any(seen)
    assert not _C.plain([x.as_subclass(type("Own", (torch.Tensor,), {}))])


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("affine", [True, False])
def test_batch_norm_affine_is_the_fp32_expression(dtype, affine):
    """Bit for bit, whatever the type of the module's tensors, which stay as they are."""
    torch.manual_seed(0)
    norm = minuet.nn.BatchNorm(37, affine=affine).to(dtype).eval()
    with torch.no_grad():
        for t in (*norm.parameters(), norm.running_mean):
            t.normal_()
        norm.running_var.uniform_(0.1, 2.0)
        before = [t.clone() for t in norm.state_dict().values()]
        scale = torch.rsqrt(norm.running_var.float() + norm.eps)
        scale = scale * norm.weight.float() if affine else scale
        shift = -norm.running_mean.float() * scale
        shift = shift + norm.bias.float() if affine else shift
        for got, wanted in zip(minuet.nn.fused.batch_norm_affine(norm), (scale, shift)):
            assert got.dtype == torch.float32 and torch.equal(got, wanted)
    assert all(torch.equal(a, b) for a, b in zip(before, norm.state_dict().values()))


def test_rules_follow_the_form_of_a_layer():
    """Both sides of each line that a stride, a dilation or the kernel's sizes move."""
    F, half, single = minuet.nn.functional, torch.float16, torch.float32
    form = F.layer_form
    assert form((1, 1), (1, 1), False) == form((1, 1), (1, 1), True) == "plain" and form((1,), (2,), False) == "dilated"
    assert form((2, 1), (1, 1), False) == "strided" and form((2, 2), (1, 1), True) == "transposed"
    assert form((3,), (1,), False) == form((2,), (2,), True) == "other"
    # 16 bits, more than 128 output channels: up to 36 offsets over any rows, 5x5x5 over few and over many
    assert all(F.prefers_implicit_over(27, 32, 256, half, rows) for rows in (100, 30000, 10 ** 6))
    assert not F.prefers_implicit(27, 32, 256, half, "other") and F.prefers_implicit(27, 32, 128, half, "other")
    assert not F.prefers_implicit(125, 32, 256, half, "other")
    for cout, kind, few in ((256, "plain", 10000), (512, "plain", 5000), (160, "strided", 10000),
                            (256, "dilated", 6000), (132, "transposed", 6000)):
        assert F.implicit_rows_few(125, 32, cout, half, kind) == few
        took = [rows for rows in (few, few + 1, 99999, 100000) if F.prefers_implicit_over(125, 32, cout, half, rows, kind)]
        assert took == [few, 100000]
    never = F.implicit_rows_limit(64, half) + 1
    assert [F.implicit_rows_from(125, 64, 160, half, kind) for kind in ("plain", "strided", "dilated", "transposed")] == [
        150000, never, never, 150000]
    assert [F.implicit_rows_from(125, 64, 256, half, kind) for kind in ("strided", "dilated", "other")] == [100000, 100000, never]
    # fp32: few input channels under odd kernels, and plain layers that come back
    for offsets, kind, all_rows in ((27, "plain", True), (75, "dilated", True), (125, "strided", True), (27, "transposed", True),
                                    (125, "transposed", False), (64, "plain", False), (27, "other", False)):
        assert F.prefers_hits(offsets, 16, 256, single, 60000, kind) == all_rows
    assert F.prefers_hits(64, 16, 256, single, 250000) and not F.prefers_hits(64, 16, 256, single, 249999)
    assert not F.prefers_hits(64, 32, 256, single, 300000) and F.prefers_hits(75, 32, 256, single, 300000)
    assert not any(F.prefers_hits(27, 32, 256, single, 10 ** 6, kind) for kind in ("dilated", "strided", "transposed", "other"))


def test_saved_layers_work_out_their_routes_anew():
    import pickle
    conv = minuet.nn.SparseConv(3, 4, 8, 3)
    conv._routes["lines", torch.float16] = 7          # as another version may have kept them
    assert pickle.loads(pickle.dumps(conv))._routes == {} and conv._routes

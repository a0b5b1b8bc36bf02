"""The forward of wide 16-bit layers whose rows and weights stream through LDS,
with and without tiles, against a plain fp32 product per offset."""
import pytest
import torch

import minuet_amd as minuet
from minuet_amd.nn import functional as F
from minuet_amd.nn.functional import _C
from test_gpu_tiles import DEVICE, close, operands, reference, tile_rows

pytestmark = pytest.mark.gpu

# one target, one more and one fewer than a workgroup's; every shape of a workgroup (32 x 64, 64 x 64,
# 128 x 64, 64 x 128, 128 x 128); rows of one to four stages, whole and ragged; outputs that are no whole
# pieces and several column blocks; fewer offsets than the ring holds, and more than a wavefront has lanes
SHAPES = [
    (1, 27, 128, 128), (33, 3, 72, 4), (500, 2, 256, 512), (1000, 125, 136, 64), (1025, 27, 64, 160),
    (2000, 27, 200, 36), (5000, 27, 128, 128), (4097, 9, 192, 100), (16500, 27, 128, 64), (20000, 8, 256, 32),
    (9000, 27, 128, 128), (8300, 33, 144, 256), (50000, 27, 128, 128), (26000, 3, 192, 160), (25700, 128, 72, 256)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("targets,offsets,cin,cout", SHAPES)
def test_forward_matches_products(targets, offsets, cin, cout, dtype):
    assert _C.streamed_forward_supported(offsets, cin, cout, dtype)
    dense, x, w = operands(targets, 3000, offsets, cin, cout, dtype)
    packed = F.pack_weights(w)
    tiles = _C.kernel_map_tiles(dense)
    wanted = reference(x, w, dense)
    plain = _C.sparse_convolution_forward_implicit(x, w, dense, packed_weights=packed)
    close(plain, wanted, dtype)
    assert torch.equal(_C.sparse_convolution_forward_tiled(x, w, tiles, targets, packed), plain)
    gen = torch.Generator(device=DEVICE).manual_seed(9)
    scale, shift = (torch.randn(cout, generator=gen, device=DEVICE) for _ in range(2))
    residual = torch.randn(targets, cout, generator=gen, device=DEVICE).to(dtype)
    epilogue = F.Epilogue(scale, shift, residual, "relu", 0.0)
    wanted = torch.relu(wanted * scale + shift + residual.float())
    plain = _C.sparse_convolution_forward_implicit(x, w, dense, epilogue=epilogue, packed_weights=packed)
    close(plain, wanted, dtype)
    assert torch.equal(_C.sparse_convolution_forward_tiled(x, w, tiles, targets, packed, epilogue=epilogue), plain)


@pytest.mark.parametrize("targets,cin,cout", [(1, 128, 64), (1000, 256, 64), (5000, 128, 128), (17000, 192, 64),
                                              (9000, 128, 128), (50000, 128, 128)])
def test_undefined_numbers_stay_where_they_belong(targets, cin, cout):
    """A weight that is not finite reaches none of the 32 targets that stand
    together where none uses its offset, a feature that is not finite the targets
    that use its row, and every other row is what it is without."""
    dense, x, w = operands(targets, 3000, 27, cin, cout, torch.float16)
    dense[[0, 5, 26]] = -1
    dense[9] = -1
    dense[9, targets // 2] = 7
    packed = F.pack_weights(w)
    tiles = _C.kernel_map_tiles(dense)
    spoilt = w.clone()
    spoilt[[0, 5, 26], 0, 3] = torch.tensor([float("inf"), float("nan"), float("-inf")], device=DEVICE).half()
    wild = spoilt.clone()
    wild[9, 1, 2] = float("inf")
    bad = x.clone()
    bad[7, 3], bad[11, cin - 1] = float("inf"), float("nan")
    touched = ((dense == 7) | (dense == 11)).any(0)
    wanted = _C.sparse_convolution_forward_implicit(x, w, dense, packed_weights=packed)
    assert bool(wanted.isfinite().all())
    places = torch.arange(-(-targets // 32) * 32, device=DEVICE)
    for at, forward in (
            (places, lambda f, weights: _C.sparse_convolution_forward_implicit(f, weights, dense)),
            (tile_rows(tiles, targets).long(),
             lambda f, weights: _C.sparse_convolution_forward_tiled(f, weights, tiles, targets, F.pack_weights(weights)))):
        assert torch.equal(forward(x, spoilt), wanted)
        groups = at.view(-1, 32)
        others = groups[~(groups == targets // 2).any(1)].flatten()
        others = others[(others >= 0) & (others < targets)]
        assert torch.equal(forward(x, wild)[others], wanted[others])
        got = forward(bad, w)
        assert torch.equal(got[~touched], wanted[~touched]) and not bool(got[touched].isfinite().all(1).any())


# strided, 3x3x3 and 5x5x5; every workgroup shape and rows of one to four stages among them
@pytest.mark.parametrize("targets,offsets,cin,cout", [
    (700, 8, 128, 256), (3000, 27, 64, 160), (5000, 27, 256, 128), (6000, 125, 136, 64), (17000, 8, 192, 96),
    (9000, 27, 128, 128), (26000, 27, 144, 128)])
def test_weights_that_are_not_finite_reach_their_targets_only(targets, offsets, cin, cout):
    """Those that have a source under the offset, one by one."""
    dense, x, w = operands(targets, 3000, offsets, cin, cout, torch.float16)
    tiles = _C.kernel_map_tiles(dense)
    plain = _C.sparse_convolution_forward_implicit(x, w, dense, packed_weights=F.pack_weights(w))
    assert bool(plain.isfinite().all())
    for offset in (0, offsets // 2, offsets - 1):
        spoilt = w.clone()
        spoilt[offset, cin - 1, 3], spoilt[offset, 0, cout - 1] = float("-inf"), float("nan")
        reached = torch.zeros(targets, cout, dtype=torch.bool, device=DEVICE)
        reached[:, [3, cout - 1]] = (dense[offset] >= 0)[:, None]
        packed = F.pack_weights(spoilt)
        for got in (_C.sparse_convolution_forward_implicit(x, spoilt, dense, packed_weights=packed),
                    _C.sparse_convolution_forward_tiled(x, spoilt, tiles, targets, packed)):
            assert torch.equal(got[~reached], plain[~reached]) and not bool(got[reached].isfinite().any())


def test_a_layer_gives_the_same_rows_from_call_to_call():
    """The first call, later ones through the extension module, one on another
    stream, which has no tiles, and the replays of a captured one."""
    from helpers import random_cloud, sorted_unique, dev
    c, _ = sorted_unique(random_cloud(9000, 40, 3, lo=-9), None)
    conv = minuet.nn.SparseConv3d(256, 256, 3, dtype=torch.float16, device=DEVICE)
    cache = minuet.nn.KernelMapCache(3, torch.int32, DEVICE)
    minuet.set_kernel_map_cache(conv, cache)
    x = minuet.SparseTensor(torch.randn(c.shape[0], 256, device=DEVICE).half(), dev(c))
    with torch.no_grad():
        first = conv(x).F
        assert [bool(entry) for entry in cache._offset_groups_cache.values()] == [True]     # tiles, kept with the map
        assert torch.equal(conv(x).F, first)
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            other = conv(x).F
        side.synchronize()
        assert torch.equal(other, first)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = conv(x).F
        for _ in range(3):
            out.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, first)


@pytest.mark.parametrize("cin,cout,offsets,streams", [
    (256, 96, 27, False), (256, 104, 27, True), (200, 96, 9, False), (192, 96, 27, True), (256, 32, 8, True),
    (128, 128, 27, True), (128, 128, 36, True), (128, 128, 45, False), (256, 128, 64, False), (192, 224, 125, False)])
def test_which_wide_layers_are_streamed(cin, cout, offsets, streams):
    """Both sides of the line between streaming and grouped products."""
    assert F.prefers_streamed(offsets, cin, cout, torch.float16) == streams


@pytest.mark.parametrize("rows,cout,dtype,streams", [(5000, 160, torch.float16, True), (5441, 160, torch.float16, False),
                                                     (9000, 160, torch.bfloat16, True), (9000, 200, torch.float16, True),
                                                     (9000, 128, torch.float16, True), (3300, 320, torch.float16, False)])
def test_how_many_rows_are_streamed(rows, cout, dtype, streams, monkeypatch):
    """Each cloud gets the kernel that a fresh cache would give it."""
    generator = torch.Generator().manual_seed(rows)
    conv = minuet.nn.SparseConv3d(256, cout, 3, dtype=dtype, device=DEVICE)
    calls = []
    for name in ("implicit", "tiled", "groups"):
        whole = getattr(_C, f"sparse_convolution_forward_{name}")
        monkeypatch.setattr(_C, f"sparse_convolution_forward_{name}",
                            lambda *args, _whole=whole, _name=name, **kw: calls.append(_name) or _whole(*args, **kw))
    wanted = {}
    for count in (rows, 700, rows, 700):
        cells = torch.randperm(1 << 15, generator=generator)[:count].sort()[0].to(DEVICE)
        coordinates = torch.stack([cells >> 10, (cells >> 5) & 31, cells & 31], 1).int()
        x = minuet.SparseTensor(torch.randn(count, 256, device=DEVICE).to(dtype), coordinates)
        conv.set_kernel_map_cache(minuet.nn.KernelMapCache(3, torch.int32, DEVICE))
        with torch.no_grad():
            conv(x)
            assert (calls[-1] == "groups") == (count == rows and not streams)
            got = conv(x).F
        wide = sum((x.F.double().new_zeros(count, cout).index_add_(0, t, x.F[s].double() @ conv.kernel[o].double())
                    for o, s, t in _pairs(coordinates)))
        # products of unit normals and uniform weights, rounded once or (grouped) twice
        assert float((got.double() - wide).norm() / wide.norm()) < 4 * torch.finfo(dtype).eps


def _pairs(coordinates):
    key = lambda c: ((c[:, 0].long() + 1) * 64 + c[:, 1] + 1) * 64 + c[:, 2] + 1
    keys = key(coordinates)
    for o, offset in enumerate(minuet.utils.helpers.generate_kernel_offsets(3, 3, 1, 1)):
        wanted = key(coordinates + torch.as_tensor(offset, device=coordinates.device, dtype=torch.int32))
        at = torch.searchsorted(keys, wanted).clamp_(max=len(keys) - 1)
        t = torch.nonzero(keys[at] == wanted)[:, 0]
        yield o, at[t], t


@pytest.mark.parametrize("cin,streams", [(96, True), (100, False), (104, True), (150, False), (254, False), (256, True)])
def test_rows_that_need_padding_are_not_streamed(cin, streams):
    conv = minuet.nn.SparseConv3d(cin, 128, 3, dtype=torch.float16, device=DEVICE)
    features = torch.empty(1, cin, dtype=torch.float16, device=DEVICE)
    pad = conv._row_padding(features)
    assert (pad == 0) == streams and conv._takes_implicit(features, pad) == streams


# in tiles, and with one source a target
@pytest.mark.parametrize("transposed", [False, True])
def test_layers_that_record_gradients_run_the_same_kernels(transposed, monkeypatch):
    from helpers import random_cloud, sorted_unique, dev
    c, _ = sorted_unique(random_cloud(70000, 48, 3, lo=-9), None)
    cache = minuet.nn.KernelMapCache(3, torch.int32, DEVICE)
    conv = minuet.nn.SparseConv(3, 256, 192, 2 if transposed else 3, stride=2 if transposed else 1, transposed=transposed,
                                dtype=torch.bfloat16, device=DEVICE)
    conv.set_kernel_map_cache(cache)
    x = minuet.SparseTensor(torch.randn(c.shape[0], 256, device=DEVICE).bfloat16(), dev(c))
    with torch.no_grad():
        if transposed:
            down = minuet.nn.SparseConv3d(256, 256, 2, stride=2, dtype=torch.bfloat16, device=DEVICE)
            down.set_kernel_map_cache(cache)
            x = down(x)
        wanted = conv(x).F
    name = "sparse_convolution_forward_" + ("single" if transposed else "tiled")
    whole, calls = getattr(_C, name), []
    monkeypatch.setattr(_C, name, lambda *args, **options: calls.append(1) or whole(*args, **options))
    for _ in range(2):
        assert torch.equal(conv(x).F.detach(), wanted)
    assert len(calls) == 2
    with torch.no_grad():
        conv.kernel.mul_(2.0)
    assert torch.equal(conv(x).F.detach(), 2 * wanted)


# one round of workgroups on 256 compute units, and two
@pytest.mark.parametrize("cout,most", [(32, 32768), (64, 32768), (96, 16384), (128, 16384), (160, 8192), (256, 8192),
                                       (320, 5440)])
def test_tiles_from_the_second_round_of_workgroups_on(cout, most):
    worth = lambda targets: _C.kernel_map_tiles_worth_making(targets, 27, 192, cout, torch.float16)
    assert not worth(most) and worth(most + 64)

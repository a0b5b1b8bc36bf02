"""The output-stationary forward with and without tiles of targets that share
their live offsets, against a plain fp32 product per offset."""
import ctypes

import pytest
import torch

import minuet_amd as minuet
from minuet_amd.nn import functional as F
from minuet_amd.nn.functional import _C
from minuet_amd.unet import SparseUNet

pytestmark = pytest.mark.gpu
DEVICE = "cuda:0"


def random_map(targets, sources, offsets, density, seed):
    """A map whose targets use few offsets each, some of them none at all."""
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    index = torch.randint(0, sources, (offsets, targets), generator=gen, device=DEVICE, dtype=torch.int32)
    liking = torch.rand(offsets, 1, generator=gen, device=DEVICE) * 2 * density
    hit = torch.rand(offsets, targets, generator=gen, device=DEVICE) < liking
    hit &= torch.rand(targets, generator=gen, device=DEVICE) > 0.1
    return torch.where(hit, index, torch.full_like(index, -1))


def reference(x, w, dense):
    kind = torch.float64 if x.dtype == torch.float64 else torch.float32
    out = torch.zeros(dense.shape[1], w.shape[2], device=x.device, dtype=kind)
    for o in range(dense.shape[0]):
        rows = x.to(kind)[dense[o].clamp(min=0).long()] * (dense[o] >= 0)[:, None]
        out += rows @ w[o].to(kind)
    return out


def operands(targets, sources, offsets, cin, cout, dtype, seed=0, density=0.3):
    gen = torch.Generator(device=DEVICE).manual_seed(seed + 1)
    dense = random_map(targets, sources, offsets, density, seed)
    x = torch.randn(sources, cin, generator=gen, device=DEVICE).to(dtype)
    w = (torch.randn(offsets, cin, cout, generator=gen, device=DEVICE) / (cin * offsets * density) ** 0.5).to(dtype)
    return dense, x, w


def close(got, wanted, dtype):
    bound = 4e-3 if dtype == torch.float16 else 2e-2
    assert float((got.float() - wanted).norm() / wanted.norm().clamp(min=1e-6)) < bound


# one target, tiles of one short of, exactly and one more than 128, several windows of 4 096 per die
@pytest.mark.parametrize("targets,offsets", [(1, 27), (127, 27), (128, 9), (1025, 27), (5000, 33), (33000, 27),
                                             (33000, 125), (2000, 128), (2000, 49), (2000, 50)])
def test_tiles_are_the_targets(targets, offsets):
    dense = random_map(targets, targets, offsets, 0.2, 5)
    tiles = _C.kernel_map_tiles(dense).cpu()
    windows = 8 * max(1, -(-targets // (8 * 4096)))
    per_window = -(--(-targets // windows) // 128)
    count = windows * per_window
    rows, counts = tiles[:count * 128].view(count, 128), tiles[count * 128:count * 129]
    offsets_at = count * 128 + -(-count // 4) * 4
    numbers = tiles[offsets_at:offsets_at + count * offsets].view(count, offsets)
    sources = tiles[offsets_at + -(-(count * offsets) // 4) * 4:].view(count, offsets, 128)
    assert torch.equal(torch.sort(rows[rows >= 0])[0], torch.arange(targets, dtype=torch.int32))
    dense = dense.cpu()
    for t in range(count):
        live, mine = int(counts[t]), rows[t]
        assert (live == 0) == bool((mine < 0).all())
        if live == 0:
            continue
        there = mine >= 0
        entries = torch.where(there, dense[:, mine.clamp(min=0).long()], torch.tensor(-1, dtype=torch.int32))
        used = torch.nonzero((entries >= 0).any(1))[:, 0].int()
        assert torch.equal(numbers[t, :live], used if used.numel() else torch.zeros(1, dtype=torch.int32))
        assert torch.equal(sources[t, :live], entries[numbers[t, :live].long()])


# rows of one, two and a ragged number of 16-byte pieces, of one stage and of several; channel
# blocks one to four and two groups; outputs that are no whole pieces; each number of workgroups
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("targets,offsets,cin,cout", [
    (1, 27, 64, 64), (129, 27, 64, 64), (5000, 27, 32, 32), (5000, 27, 24, 12), (5000, 8, 16, 96), (20000, 27, 48, 64),
    (20000, 2, 72, 128), (3000, 27, 128, 160), (3000, 33, 200, 36), (40000, 27, 64, 96), (66000, 9, 64, 128),
    (90000, 27, 32, 32), (90000, 27, 40, 64), (300000, 3, 64, 64), (2000, 125, 64, 32)])
def test_forward_matches_products(targets, offsets, cin, cout, dtype):
    dense, x, w = operands(targets, 3000, offsets, cin, cout, dtype)
    packed = F.pack_weights(w)
    wanted = reference(x, w, dense)
    close(_C.sparse_convolution_forward_implicit(x, w, dense, packed_weights=packed), wanted, dtype)
    tiles = _C.kernel_map_tiles(dense)
    close(_C.sparse_convolution_forward_tiled(x, w, tiles, targets, packed), wanted, dtype)
    gen = torch.Generator(device=DEVICE).manual_seed(9)
    scale, shift = (torch.randn(cout, generator=gen, device=DEVICE) for _ in range(2))
    residual = torch.randn(targets, cout, generator=gen, device=DEVICE).to(dtype)
    epilogue = F.Epilogue(scale, shift, residual, "relu", 0.0)
    wanted = torch.relu(wanted * scale + shift + residual.float())
    close(_C.sparse_convolution_forward_implicit(x, w, dense, epilogue=epilogue, packed_weights=packed), wanted, dtype)
    close(_C.sparse_convolution_forward_tiled(x, w, tiles, targets, packed, epilogue=epilogue), wanted, dtype)


def tile_rows(tiles, targets):
    """The targets of every tile's places (-1: none), as test_tiles_are_the_targets reads them."""
    windows = 8 * max(1, -(-targets // (8 * 4096)))
    return tiles[:windows * -(--(-targets // windows) // 128) * 128]


# both stage forms (two offsets of rows of 64 bytes, one of wider ones), one and two sets of wavefronts,
# the kernel for large maps, and tiles whose lanes load alone and together
@pytest.mark.parametrize("cin", [32, 64])
@pytest.mark.parametrize("targets", [1, 3000, 60000, 70000, 90000])
def test_undefined_weights_stay_with_their_offsets(targets, cin):
    """A weight that is not finite reaches the 32 targets of a wavefront that uses
    its offset, and no others: with it at offsets that nobody uses (the first,
    the last, one between) every row is what it is without, and with it where one
    target uses it the rows outside that target's wavefront are."""
    dense, x, w = operands(targets, 3000, 27, cin, 64, torch.float16)
    dense[[0, 5, 26]] = -1
    dense[9] = -1
    dense[9, targets // 2] = 7
    spoilt = w.clone()
    spoilt[[0, 5, 26], 0, 3] = torch.tensor([float("inf"), float("nan"), float("-inf")], device=DEVICE).half()
    wild = spoilt.clone()
    wild[9, 1, 2] = float("inf")
    tiles = _C.kernel_map_tiles(dense)
    place = tile_rows(tiles, targets).long()
    plain = torch.arange(-(-targets // 32) * 32, device=DEVICE)

    def rows_without(places):
        groups = places.view(-1, 32)
        return groups[~(groups == targets // 2).any(1)].flatten()

    for forward, places in (
            (lambda weights: _C.sparse_convolution_forward_implicit(x, weights, dense), plain),
            (lambda weights: _C.sparse_convolution_forward_tiled(x, weights, tiles, targets, F.pack_weights(weights)), place)):
        wanted = forward(w)
        assert bool(wanted.isfinite().all())
        assert torch.equal(forward(spoilt), wanted)
        others = rows_without(places)
        others = others[(others >= 0) & (others < targets)]
        assert torch.equal(forward(wild)[others], wanted[others])


def scattered_cloud():
    gen = torch.Generator(device=DEVICE).manual_seed(3)
    cells = torch.randperm(1 << 20, generator=gen, device=DEVICE)[:100000]
    coordinates = torch.stack([cells >> 13, (cells >> 6) & 127, cells & 63], 1).int()
    return coordinates[F.build_sorted_index(coordinates)], gen


@pytest.mark.parametrize("cin,cout,dtype", [(64, 64, torch.float16), (32, 32, torch.bfloat16), (24, 96, torch.float16),
                                            (128, 64, torch.float16)])
def test_layer_comes_to_use_tiles(cin, cout, dtype):
    """A map that is read on and on gets tiles; the layer's results stay bit for bit."""
    coordinates, gen = scattered_cloud()
    conv = minuet.nn.SparseConv3d(cin, cout, 3, dtype=dtype, device=DEVICE)
    minuet.set_kernel_map_cache(conv, minuet.nn.KernelMapCache(3, torch.int32, DEVICE))
    x = minuet.SparseTensor(torch.randn(100000, cin, generator=gen, device=DEVICE).to(dtype), coordinates)
    with torch.no_grad():
        first = conv(x).F
        held = torch.cuda.memory_allocated()
        for _ in range(60):
            last = conv(x).F
        assert torch.cuda.memory_allocated() > held + 100000 * 27 * 4      # the tiles
    assert torch.equal(last, first)


@pytest.mark.parametrize("cin,cout,dtype", [(4, 32, torch.float16), (8, 64, torch.bfloat16), (32, 32, torch.float32)])
def test_layers_that_take_no_tiles_share_a_map_that_has_them(cin, cout, dtype):
    """The map belongs to its kernel size and stride: once a wide layer has earned
    it tiles, a stem or an fp32 layer over it runs as before."""
    coordinates, gen = scattered_cloud()
    wide = minuet.nn.SparseConv3d(64, 64, 3, dtype=torch.float16, device=DEVICE)
    conv = minuet.nn.SparseConv3d(cin, cout, 3, dtype=dtype, device=DEVICE)
    cache = minuet.nn.KernelMapCache(3, torch.int32, DEVICE)
    for module in (wide, conv):
        minuet.set_kernel_map_cache(module, cache)
    x = minuet.SparseTensor(torch.randn(100000, cin, generator=gen, device=DEVICE).to(dtype), coordinates)
    y = minuet.SparseTensor(torch.randn(100000, 64, generator=gen, device=DEVICE).half(), coordinates)
    with torch.no_grad():
        first = conv(x).F
        for _ in range(20):
            wide(y)
            again = conv(x).F
    assert torch.equal(again, first)


def test_network_on_kept_maps():
    """Ten passes over the same maps, and a captured one, equal the first."""
    coordinates, gen = scattered_cloud()
    torch.manual_seed(0)
    net = SparseUNet(4, 32, dtype=torch.float16, device=DEVICE).eval()
    minuet.set_kernel_map_cache(net, minuet.nn.KernelMapCache(3, torch.int32, DEVICE))
    x = minuet.SparseTensor(torch.randn(100000, 4, generator=gen, device=DEVICE).half(), coordinates)
    with torch.no_grad():
        first = net(x).F
        for _ in range(9):
            assert torch.equal(net(x).F, first)
    graphed = minuet.capture_forward(lambda: net(x))
    for _ in range(3):
        assert torch.equal(graphed.replay().F, first)


def test_tiles_made_on_one_stream_and_read_on_another():
    """The tiles' store addresses are read by other streams only when they are
    written, and stay theirs until their last reader is done."""
    coordinates, gen = scattered_cloud()
    conv = minuet.nn.SparseConv3d(64, 64, 3, dtype=torch.float16, device=DEVICE)
    cache = minuet.nn.KernelMapCache(3, torch.int32, DEVICE)
    minuet.set_kernel_map_cache(conv, cache)
    x = minuet.SparseTensor(torch.randn(100000, 64, generator=gen, device=DEVICE).half(), coordinates)
    lib = _C.load_library()
    size = ctypes.c_int64()
    assert lib.mnt_kernel_map_tiles_size(100000, 27, ctypes.byref(size)) == 0
    maker, reader = torch.cuda.Stream(), torch.cuda.Stream()
    with torch.no_grad():
        first = conv(x).F
        held = torch.cuda.memory_allocated()
        torch.cuda.synchronize()
        with torch.cuda.stream(maker):
            torch.cuda._sleep(2_000_000)                 # the tiles are far from written when the other stream calls
            for _ in range(60):
                conv(x)
                if torch.cuda.memory_allocated() >= held + 4 * size.value:
                    break
        assert torch.cuda.memory_allocated() >= held + 4 * size.value
        with torch.cuda.stream(reader):
            assert torch.equal(conv(x).F, first)
        torch.cuda.synchronize()
        with torch.cuda.stream(reader):                  # with tiles now, read late, after the cache has let go of them
            torch.cuda._sleep(2_000_000)
            last = conv(x).F
        cache.reset()
        with torch.cuda.stream(maker):
            taken = [torch.zeros(size.value, dtype=torch.int32, device=DEVICE) for _ in range(3)]
        torch.cuda.synchronize()
    assert torch.equal(last, first) and len(taken) == 3


@pytest.mark.parametrize("targets", [1, 129, 32769, 7 * 32768 + 1, 16 * 32768 + 77])
def test_every_target_has_one_place(targets):
    """One window of tiles per die, several, more than a band of them and two
    bands with a remainder: every target stands in one tile, and the tiles of
    the smallest numbers are a window's longest."""
    gen = torch.Generator(device="cuda").manual_seed(targets)
    dense = torch.randint(0, targets, (9, targets), generator=gen, device="cuda", dtype=torch.int32)
    dense[torch.rand(9, targets, generator=gen, device="cuda") < 0.8] = -1
    windows = 8 * max(1, -(-targets // 32768))
    window = -(-max(1, -(-targets // windows)) // 128) * 128
    tiles = windows * window // 128
    packed = _C.kernel_map_tiles(dense)
    rows = packed[:tiles * 128].view(tiles, 128)
    counts = packed[tiles * 128:tiles * 128 + tiles]
    assert rows[rows >= 0].sort().values.equal(torch.arange(targets, device="cuda", dtype=torch.int32))
    used = rows.amax(1) >= 0
    assert (counts > 0).equal(used)
    owner = torch.where(used, rows.amax(1) // window, -1)
    assert (owner[used] % 8).equal(torch.arange(tiles, device="cuda", dtype=torch.int32)[used] % 8)
    for w in range(0, windows, max(1, windows // 5)):
        mine = counts[owner == w]
        assert mine.equal(mine.sort(descending=True).values)


def test_planned_passes_make_the_tiles_of_all_maps_together():
    """From the pass after the first planned one on: the same rows, from tiles that
    are there before the first layer; a pass over a cloud too small for them has none."""
    coordinates, gen = scattered_cloud()
    torch.manual_seed(0)
    layers = [minuet.nn.SparseConv3d(64, 64, 3, dtype=torch.float16, device=DEVICE) for _ in range(5)]
    layers += [minuet.nn.SparseConv3d(64, 64, 2, stride=2, dtype=torch.float16, device=DEVICE)]
    net = torch.nn.Sequential(*layers)
    cache = minuet.nn.KernelMapCache(3, torch.int32, DEVICE)
    minuet.set_kernel_map_cache(net, cache)
    features = torch.randn(100000, 64, generator=gen, device=DEVICE).half()

    def run(rows):
        cache.reset()
        out = net(minuet.SparseTensor(features[:rows], coordinates[:rows].contiguous())).F
        return out, len(cache._built.tiles) if cache._built is not None else -1

    with torch.no_grad():
        first, _ = run(100000)
        made = []
        for _ in range(4):
            again, tiles = run(100000)
            made.append(tiles)
            assert torch.equal(again, first)
        assert made[0] <= 0 < made[-1]
        small = [run(500)[0] for _ in range(4)]
        assert cache._built.tiles == {} and all(torch.equal(s, small[0]) for s in small)
        again, _ = run(100000)
        assert torch.equal(again, first)


@pytest.mark.parametrize("count", [1, 8, 9])
def test_tiles_of_several_maps_at_once(count):
    """One set of launches, and two; maps of up to 32 offsets and of more; windows
    of one, two and four rounds of a workgroup."""
    maps = [random_map(targets, 700, offsets, 0.3, targets + offsets).cuda()
            for targets, offsets in ((9000, 27), (300, 27), (4100, 8), (130, 40), (40000, 27), (70, 125), (1, 2),
                                     (20000, 27), (1000, 33))[:count]]
    together = _C.kernel_maps_tiles([(m.data_ptr(), m.shape[1], m.shape[0]) for m in maps], torch.device(DEVICE))
    for dense, tiles in zip(maps, together):
        alone = _C.kernel_map_tiles(dense)
        x, w = operands_of(dense)
        assert _C.sparse_convolution_forward_tiled(x, w, tiles, dense.shape[1], F.pack_weights(w)).equal(
            _C.sparse_convolution_forward_tiled(x, w, alone, dense.shape[1], F.pack_weights(w)))


def operands_of(dense):
    gen = torch.Generator(device=DEVICE).manual_seed(1)
    return (torch.randn(700, 32, generator=gen, device=DEVICE).half(),
            torch.randn(dense.shape[0], 32, 32, generator=gen, device=DEVICE).half())


@pytest.mark.parametrize("first", ["wide", "narrow"])
def test_layers_of_one_map_make_its_tiles_once(first):
    """Whichever asks for them, and whichever of the others describes the map to the
    extension module after that."""
    cells = torch.randperm(1 << 18, generator=torch.Generator().manual_seed(4))[:70000].cuda()
    coordinates = torch.stack([cells >> 12, (cells >> 6) & 63, cells & 63], 1).int()
    coordinates = coordinates[F.build_sorted_index(coordinates)]
    cache = minuet.nn.KernelMapCache(3, torch.int32, "cuda")
    layers = {width: minuet.nn.SparseConv3d(width, width, 3, dtype=torch.float16, device="cuda") for width in (128, 64, 32)}
    inputs = {width: minuet.SparseTensor(torch.randn(len(coordinates), width, device="cuda").half(), coordinates)
              for width in layers}
    for layer in layers.values():
        layer.set_kernel_map_cache(cache)
    with torch.no_grad():
        def run(width):
            return layers[width](inputs[width]).F.double().sum().item()
        wanted = {}
        for width in (128, 64) if first == "wide" else (64, 128):
            wanted[width] = run(width)
            for _ in range(30):
                run(width)
        entry, = (entry for maps in cache._fast_maps.values() for entry in maps.values())
        saved = entry.tiles_saved
        assert saved > 0
        torch.cuda.synchronize()
        before = torch.cuda.memory_allocated()
        for _ in range(3):
            for width in (128, 64):
                assert run(width) == wanted[width]
        run(32)                                              # (describes the map once more)
        weights = torch.cuda.memory_allocated() - before
        for _ in range(30):
            for width in (128, 64, 32):
                run(width)
        assert torch.cuda.memory_allocated() - before <= weights < 1 << 20       # (tiles take 8 MB)
        kept, = (entry for maps in cache._fast_maps.values() for entry in maps.values())
        assert kept is entry and kept.tiles_saved > saved


# the kernel for few targets with one and two sets of wavefronts, the one for many, tiles of both; one to four
# groups of channels, a last one of less than a block; rows of 16 to 64 bytes
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("targets,offsets,cin,cout", [
    (1, 27, 32, 132), (3000, 27, 8, 512), (700, 8, 24, 160), (60000, 27, 16, 256), (70000, 27, 32, 132), (90000, 8, 24, 384),
    (5000, 125, 32, 160), (66000, 125, 8, 136)])
def test_weights_that_are_not_finite_under_many_channels(targets, offsets, cin, cout, dtype):
    """Rows of up to 64 bytes and more than 128 output channels, which three kernels took before: a weight that is
    not finite reaches the targets that have a source under its offset, one by one."""
    dense, x, w = operands(targets, 3000, offsets, cin, cout, dtype)
    tiles = _C.kernel_map_tiles(dense)
    spoilt = w.clone()
    reached = torch.zeros(targets, cout, dtype=torch.bool, device=DEVICE)
    for offset, value in ((0, "inf"), (offsets // 2, "nan"), (offsets - 1, "-inf")):
        spoilt[offset, cin - 1, 3], spoilt[offset, 0, cout - 1] = float(value), float(value)
        reached[:, [3, cout - 1]] |= (dense[offset] >= 0)[:, None]
    wanted = reference(x, w, dense)
    size = reference(x.abs(), w.abs(), dense)
    # sums of up to 125 x 32 products in 32 bits, in whichever order, and one rounding
    bound = torch.finfo(dtype).eps * wanted.abs() + 2 * offsets * cin * 2.0 ** -24 * size + 1e-7
    plain = [_C.sparse_convolution_forward_implicit(x, w, dense), _C.sparse_convolution_forward_tiled(
        x, w, tiles, targets, F.pack_weights(w))]
    got = [_C.sparse_convolution_forward_implicit(x, spoilt, dense), _C.sparse_convolution_forward_tiled(
        x, spoilt, tiles, targets, F.pack_weights(spoilt))]
    for before, after in zip(plain, got):
        assert bool(((before.float() - wanted).abs() <= bound).all())
        assert not bool(after[reached].isfinite().any())
        assert bool(((after.float() - wanted).abs() <= bound)[~reached].all())
        untouched = torch.ones(cout, dtype=torch.bool, device=DEVICE)
        untouched[[3, cout - 1]] = False
        assert torch.equal(after[:, untouched], before[:, untouched])
    gen = torch.Generator(device=DEVICE).manual_seed(4)
    scale, shift = (torch.randn(cout, generator=gen, device=DEVICE) for _ in range(2))
    residual = torch.randn(targets, cout, generator=gen, device=DEVICE).to(dtype)
    for act, slope in (("relu", 0.0), ("leaky_relu", 0.25), (None, 0.0)):
        epilogue = F.Epilogue(scale, shift, residual, act, slope)
        finished = wanted * scale + shift + residual
        finished = torch.where(finished > 0, finished, finished * slope) if act else finished
        limit = torch.finfo(dtype).eps * finished.abs() + scale.abs() * bound + 4 * 2.0 ** -24 * (
            scale.abs() * wanted.abs() + shift.abs() + residual.abs()) + 1e-7
        for after in (_C.sparse_convolution_forward_implicit(x, spoilt, dense, epilogue=epilogue),
                      _C.sparse_convolution_forward_tiled(x, spoilt, tiles, targets, F.pack_weights(spoilt), epilogue=epilogue)):
            assert bool(((after.float() - finished).abs() <= limit)[~reached].all())

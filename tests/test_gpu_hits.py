"""The fp32 single-kernel forward, which multiplies hits only."""
import pytest
import torch

import minuet_amd as minuet
from minuet_amd.nn import functional as F
from minuet_amd.nn.functional import _C

from test_gpu_tiles import DEVICE, operands, reference

pytestmark = pytest.mark.gpu


# targets about a workgroup's 16, 32 and 64; K of one to four pieces of 16, ragged, and more than one unit;
# N in one, two and four blocks and less than one; offsets fewer and more than a wavefront lists at once
@pytest.mark.parametrize("targets,offsets,cin,cout", [
    (1, 27, 4, 4), (63, 2, 16, 16), (65, 27, 32, 32), (1000, 8, 20, 36), (1000, 27, 48, 64), (700, 125, 32, 20),
    (15, 27, 64, 16), (17, 27, 64, 64), (1500, 27, 64, 32), (3000, 27, 32, 64), (6000, 27, 64, 64),
    (3000, 27, 100, 64), (500, 33, 256, 128), (30000, 27, 64, 64), (30000, 9, 64, 96), (70000, 27, 12, 32)])
def test_forward_matches_products(targets, offsets, cin, cout):
    dense, x, w = operands(targets, 3000, offsets, cin, cout, torch.float32)
    wanted = reference(x.double(), w.double(), dense)

    def check(got, wanted):
        assert float((got.double() - wanted).norm() / wanted.norm().clamp(min=1e-6)) < 1e-6

    out = _C.sparse_convolution_forward_implicit(x, w, dense)
    check(out, wanted)
    assert torch.equal(out, _C.sparse_convolution_forward_implicit(x, w, dense))
    gen = torch.Generator(device=DEVICE).manual_seed(9)
    scale, shift = (torch.randn(cout, generator=gen, device=DEVICE) for _ in range(2))
    residual = torch.randn(targets, cout, generator=gen, device=DEVICE)
    epilogue = F.Epilogue(scale, shift, residual, "relu", 0.0)
    check(_C.sparse_convolution_forward_implicit(x, w, dense, epilogue=epilogue),
          torch.relu(wanted * scale + shift + residual))


def test_layer_takes_it_by_size():
    assert F.prefers_hits(27, 32, 32, torch.float32, 10 ** 6) and F.prefers_hits(27, 64, 64, torch.float32, 12000)
    assert not F.prefers_hits(27, 64, 64, torch.float32, 30000)
    assert not F.prefers_hits(27, 30, 32, torch.float32, 100) and not F.prefers_hits(1, 32, 32, torch.float32, 100)
    gen = torch.Generator(device=DEVICE).manual_seed(3)
    conv = minuet.nn.SparseConv3d(64, 64, 3, dtype=torch.float32, device=DEVICE)
    results = []
    for rows, tables in ((2000, 0), (40000, 1)):
        cells = torch.randperm(1 << 16, generator=gen, device=DEVICE)[:rows]
        coordinates = torch.stack([cells >> 10, (cells >> 5) & 31, cells & 31], 1).int()
        coordinates = coordinates[F.build_sorted_index(coordinates)]
        cache = minuet.nn.KernelMapCache(3, torch.int32, DEVICE)
        minuet.set_kernel_map_cache(conv, cache)
        x = minuet.SparseTensor(torch.randn(rows, 64, generator=gen, device=DEVICE), coordinates)
        with torch.no_grad():
            out = conv(x).F
            assert torch.equal(conv(x).F, out)
        assert len(cache._kernel_maps_cache) == tables
        dense, _ = _C.kernel_map_dense(coordinates, coordinates, cache._kernel_offsets((1, 1, 1), (3, 3, 3), (1, 1, 1)), None, None)
        wanted = reference(x.F.double(), conv.kernel.detach().double(), dense)
        results.append(float((out.double() - wanted).norm() / wanted.norm()))
    assert max(results) < 1e-6


def test_kernel_follows_the_size_of_each_cloud():
    """One layer and one cache over small, large and small clouds again: every one
    runs the kernel that a fresh cache gives it, its second pass too, in each
    order and from a plan that the cloud before has left."""
    gen = torch.Generator(device=DEVICE).manual_seed(4)
    torch.manual_seed(0)
    conv = minuet.nn.SparseConv3d(64, 64, 3, dtype=torch.float32, device=DEVICE)
    inputs = []
    for rows in (2000, 40000):
        cells = torch.randperm(1 << 16, generator=gen, device=DEVICE)[:rows]
        coordinates = torch.stack([cells >> 10, (cells >> 5) & 31, cells & 31], 1).int()
        coordinates = coordinates[F.build_sorted_index(coordinates)]
        x = minuet.SparseTensor(torch.randn(rows, 64, generator=gen, device=DEVICE), coordinates)
        minuet.set_kernel_map_cache(conv, minuet.nn.KernelMapCache(3, torch.int32, DEVICE))
        conv.invalidate_cached_weights()
        with torch.no_grad():
            inputs.append((x, conv(x).F))
    cache = minuet.nn.KernelMapCache(3, torch.int32, DEVICE)
    minuet.set_kernel_map_cache(conv, cache)
    conv.invalidate_cached_weights()
    with torch.no_grad():
        for large in (0, 0, 1, 1, 0, 1, 0, 0):
            x, expected = inputs[large]
            cache.reset()
            assert torch.equal(conv(x).F, expected)      # bit for bit: the two kernels add up in different orders
            assert torch.equal(conv(x).F, expected)


@pytest.mark.parametrize("rows, targets, cin, cout", [
    (60000, 1, 16, 96), (60000, 65, 20, 68), (45000, 333, 48, 64), (52000, 129, 48, 36), (30000, 5003, 16, 256),
    (60000, 13001, 28, 96), (80000, 64, 4, 512)])
def test_products_are_added_after_in_large_layers(rows, targets, cin, cout):
    """Few input channels over so many rows that three kernels would take the layer otherwise."""
    assert rows * cin * cout > 2_100_000_000 // 27
    gen = torch.Generator(device=DEVICE).manual_seed(rows + cout)
    x = torch.randn(rows, cin, generator=gen, device=DEVICE)
    w = torch.randn(27, cin, cout, generator=gen, device=DEVICE)
    dense = torch.randint(-rows, rows, (27, targets), generator=gen, device=DEVICE, dtype=torch.int32).clamp(min=-1)
    x[int(dense[3].max())] = 0.0
    wanted, size = (torch.zeros(targets, cout, dtype=torch.float64, device=DEVICE) for _ in range(2))
    for offset in range(27):
        hit = (dense[offset] >= 0).nonzero()[:, 0]
        picked, weight = x[dense[offset, hit].long()].double(), w[offset].double()
        wanted[hit] += picked @ weight
        size[hit] += picked.abs() @ weight.abs()
    out = _C.sparse_convolution_forward_implicit(x, w, dense)
    # every value is rounded in at most cin additions of an offset and 27 + 4 of offsets and wavefronts
    assert bool(((out.double() - wanted).abs() <= (cin + 31) * 2.0 ** -24 * size).all())
    assert torch.equal(out, _C.sparse_convolution_forward_implicit(x, w, dense))
    w[5, 0, 0] = float("inf")                            # what a target has no source for does not reach it
    out = _C.sparse_convolution_forward_implicit(x, w, dense)
    assert bool(out[dense[5] < 0].isfinite().all())


@pytest.mark.parametrize("kernel, cin, cout", [(3, 3, 32), (3, 1, 4), (2, 3, 64), (5, 2, 48)])
def test_layers_of_less_than_four_channels(kernel, cin, cout):
    """Rows of less than four values are padded to four, at the first call and from the second on."""
    gen = torch.Generator(device=DEVICE).manual_seed(cin)
    torch.manual_seed(cin)
    conv = minuet.nn.SparseConv3d(cin, cout, kernel, dtype=torch.float32, device=DEVICE, bias=True)
    for rows in (1, 700, 6000):
        cells = torch.randperm(1 << 16, generator=gen, device=DEVICE)[:rows]
        coordinates = torch.stack([cells >> 10, (cells >> 5) & 31, cells & 31], 1).int()
        coordinates = coordinates[F.build_sorted_index(coordinates)]
        cache = minuet.nn.KernelMapCache(3, torch.int32, DEVICE)
        minuet.set_kernel_map_cache(conv, cache)
        dense, _ = _C.kernel_map_dense(coordinates, coordinates,
                                       cache._kernel_offsets((1, 1, 1), (kernel,) * 3, (1, 1, 1)), None, None)
        with torch.no_grad():
            for turn in range(3):
                conv.kernel.mul_(-0.5)
                x = minuet.SparseTensor(torch.randn(rows, cin, generator=gen, device=DEVICE), coordinates)
                out = conv(x).F
                wanted = reference(x.F.double(), conv.kernel.double(), dense)
                size = reference(x.F.abs().double(), conv.kernel.abs().double(), dense) + conv.bias.abs()
                # a value is rounded at most cin x offsets times in its sums and twice at the end
                bound = (cin * kernel ** 3 + 16) * 2.0 ** -24 * size
                assert bool(((out.double() - wanted - conv.bias.double()).abs() <= bound).all())
        assert len(cache._kernel_maps_cache) == 0 and conv._fast is not None


@pytest.mark.parametrize("kernel, cin, cout, rows", [(3, 1, 32, 20000), (3, 2, 64, 20000), (3, 3, 64, 20000), (2, 3, 16, 20000),
                                                     (5, 3, 32, 6000), (3, 3, 256, 50000)])
def test_padded_layers_are_as_exact_as_three_kernels(kernel, cin, cout, rows):
    """Against 64 bits.  Over 99 layers of three kinds of scene the errors are 0.81 to 1.02 times as large; of the
    320 000 values and more that there are here the norm of the error scatters by 1 / sqrt(2 x 320 000) < 0.2 %."""
    gen = torch.Generator(device=DEVICE).manual_seed(rows + cin)
    torch.manual_seed(cout)
    conv = minuet.nn.SparseConv3d(cin, cout, kernel, dtype=torch.float32, device=DEVICE)
    cells = torch.randperm(1 << 18, generator=gen, device=DEVICE)[:rows]
    coordinates = torch.stack([cells >> 12, (cells >> 6) & 63, cells & 63], 1).int()
    coordinates = coordinates[F.build_sorted_index(coordinates)]
    x = minuet.SparseTensor(torch.randn(rows, cin, generator=gen, device=DEVICE), coordinates)
    errors = []
    for flow in ("auto", "gather_gemm_scatter"):
        conv._tunable_config["dataflow"] = flow
        cache = minuet.nn.KernelMapCache(3, torch.int32, DEVICE)
        minuet.set_kernel_map_cache(conv, cache)
        with torch.no_grad():
            out = conv(x).F
        assert len(cache._kernel_maps_cache) == (flow != "auto")
        dense, _ = _C.kernel_map_dense(coordinates, coordinates, cache._kernel_offsets((1, 1, 1), (kernel,) * 3, (1, 1, 1)),
                                       None, None)
        wanted = reference(x.F.double(), conv.kernel.detach().double(), dense)
        errors.append(float((out.double() - wanted).norm() / wanted.norm()))
    assert errors[0] <= 1.03 * errors[1]


def test_padded_layers_keep_their_weights_until_told():
    """Weights of less than four input channels are kept padded: they follow what leaves a mark on the parameter,
    and a write through .data once the layer is told of it.  (Of four channels the parameter itself is read.)"""
    for cin, sees in ((3, False), (4, True)):
        gen = torch.Generator(device=DEVICE).manual_seed(cin)
        conv = minuet.nn.SparseConv3d(cin, 32, 3, dtype=torch.float32, device=DEVICE)
        minuet.set_kernel_map_cache(conv, minuet.nn.KernelMapCache(3, torch.int32, DEVICE))
        cells = torch.randperm(1 << 15, generator=gen, device=DEVICE)[:3000]
        coordinates = torch.stack([cells >> 10, (cells >> 5) & 31, cells & 31], 1).int()
        coordinates = coordinates[F.build_sorted_index(coordinates)]
        x = minuet.SparseTensor(torch.randn(3000, cin, generator=gen, device=DEVICE), coordinates)
        with torch.no_grad():
            before = [conv(x).F for _ in range(2)][1]
            conv.kernel.mul_(2.0)
            assert torch.equal(conv(x).F, 2.0 * before)
            conv(x)
            conv.kernel.data.mul_(2.0)
            assert torch.equal(conv(x).F, (4.0 if sees else 2.0) * before)
            conv.invalidate_cached_weights()
            assert torch.equal(conv(x).F, 4.0 * before) and torch.equal(conv(x).F, 4.0 * before)


@pytest.mark.parametrize("dtype, kernel, cin, cout, sizes", [
    (torch.float32, 3, 32, 64, (10000, 60000, 260000)),      # hits, product rows, hits again
    (torch.float16, 5, 64, 256, (1000, 101000)),             # product rows, one kernel
    (torch.float32, 3, 64, 64, (2000, 40000))])              # hits, product rows
def test_layers_for_every_size_are_kept(dtype, kernel, cin, cout, sizes):
    """A layer that has seen clouds of every range of rows goes through no Python code for any of them, in any
    order, also after its weights have changed and been seen by all."""
    gen = torch.Generator(device=DEVICE).manual_seed(11)
    torch.manual_seed(1)
    conv = minuet.nn.SparseConv3d(cin, cout, kernel, dtype=dtype, device=DEVICE)
    inputs = []
    for rows in sizes:
        cells = torch.randperm(1 << 21, generator=gen, device=DEVICE)[:rows]
        coordinates = torch.stack([cells >> 14, (cells >> 7) & 127, cells & 127], 1).int()
        coordinates = coordinates[F.build_sorted_index(coordinates)]
        x = minuet.SparseTensor(torch.randn(rows, cin, generator=gen, device=DEVICE).to(dtype), coordinates)
        inputs.append((x, minuet.nn.KernelMapCache(3, torch.int32, DEVICE)))
    came = []
    keep = conv._keep_fast
    conv._keep_fast = lambda *args: (came.append(args[0][0]), keep(*args))
    with torch.no_grad():
        for turn in range(2):
            wanted = []
            for x, cache in inputs:
                minuet.set_kernel_map_cache(conv, cache)
                wanted.append(conv(x).F)
            assert len(came) == len(sizes)
            for at in (*range(len(sizes)), *range(len(sizes) - 1, -1, -1), 0, len(sizes) - 1):
                x, cache = inputs[at]
                minuet.set_kernel_map_cache(conv, cache)
                assert torch.equal(conv(x).F, wanted[at])
            assert len(came) == len(sizes)
            came.clear()
            conv.kernel.mul_(-0.5)

"""Layer calls from the second on, which take the extension module's way."""
import numpy as np
import pytest
import torch
import torch.nn.utils.parametrize
import torch.nn.utils.prune as prune

import minuet_amd as minuet
from helpers import dev, random_cloud, sorted_unique
from minuet_amd.nn import functional as F
from minuet_amd.nn.functional import _C
from minuet_amd.unet import SparseUNet

pytestmark = pytest.mark.gpu
DEVICE = torch.device("cuda:0")


def layer_and_input(rows, cin, cout, dtype, seed=3, **options):
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    cells = torch.randperm(1 << 18, generator=gen, device=DEVICE)[:rows]
    coordinates = torch.stack([cells >> 12, (cells >> 6) & 63, cells & 63], 1).int()
    coordinates = coordinates[F.build_sorted_index(coordinates)]
    torch.manual_seed(seed)
    conv = minuet.nn.SparseConv3d(cin, cout, 3, dtype=dtype, device=DEVICE, **options)
    minuet.set_kernel_map_cache(conv, minuet.nn.KernelMapCache(3, torch.int32, DEVICE))
    features = torch.randn(rows, cin, generator=gen, device=DEVICE).to(dtype)
    return conv, minuet.SparseTensor(features, coordinates)


def test_no_memory_left_is_an_exception():
    """A caller that catches it and tries a smaller batch goes on."""
    conv, x = layer_and_input(200000, 32, 512, torch.float16)
    with torch.no_grad():
        first = conv(x).F
        assert torch.equal(conv(x).F, first)
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        total = torch.cuda.get_device_properties(DEVICE).total_memory
        try:
            torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (16 << 20)) / total)
            with pytest.raises(torch.cuda.OutOfMemoryError):
                conv(x)
        finally:
            torch.cuda.set_per_process_memory_fraction(1.0)
        assert torch.equal(conv(x).F, first)


class Twice(torch.nn.Module):
    def forward(self, kernel):
        return 2 * kernel


@pytest.mark.parametrize("made_by", ["prune kernel", "prune bias", "weight_norm", "parametrization"])
def test_parameters_made_from_others(made_by):
    """Call after call, and after what they are made from has changed."""
    conv, x = layer_and_input(3000, 32, 32, torch.float16, bias=True)
    plain, _ = layer_and_input(3000, 32, 32, torch.float16, bias=True)
    conv(x)
    conv(x)                                              # (a Layer is there when the parameter goes)
    if made_by == "weight_norm":
        torch.nn.utils.weight_norm(conv, "kernel")
    elif made_by == "parametrization":
        torch.nn.utils.parametrize.register_parametrization(conv, "kernel", Twice())
    else:
        prune.identity(conv, made_by.split()[1])
    with torch.no_grad():
        for step in range(3):
            if step == 1:
                source = {"prune kernel": "kernel_orig", "prune bias": "bias_orig", "weight_norm": "kernel_g"}.get(made_by)
                part = conv.parametrizations.kernel.original if source is None else getattr(conv, source)
                part.mul_(3.0)
            results = [conv(x).F for _ in range(3)]
            plain.kernel.copy_(conv.kernel)
            plain.bias.copy_(conv.bias)
            plain._kernel_map_cache.reset()
            for y in results:
                assert torch.equal(y, plain(x).F)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_bias_is_read_at_every_call(dtype):
    """Also one written through ``.data``, which marks nothing."""
    conv, x = layer_and_input(3000, 32, 32, dtype, bias=True)
    with torch.no_grad():
        conv(x)
        assert conv._fast is not None
        for step in range(3):
            conv.bias.data.copy_(torch.randn(32, device=DEVICE))
            again = conv(x).F
            conv.invalidate_cached_weights()
            assert torch.equal(again, conv(x).F)


def test_network_without_the_extension_module(monkeypatch):
    """The Python code alone: first pass, a pass from a plan, kept maps."""
    torch.manual_seed(0)
    net = SparseUNet(4, 16, dtype=torch.float16, device=DEVICE).eval()
    c, bd = sorted_unique(random_cloud(3000, 30, 1, lo=-9), np.array([0, 1000, 3000], dtype=np.int32))
    x = minuet.SparseTensor(torch.randn(c.shape[0], 4, device=DEVICE).half(), dev(c), batch_dims=dev(bd))

    def passes():
        cache = minuet.nn.KernelMapCache(3, torch.int32, DEVICE)
        minuet.set_kernel_map_cache(net, cache)
        with torch.no_grad():
            results = []
            for _ in range(2):
                cache.reset()
                results += [net(x).F, net(x).F]
        return results

    with_it = passes()
    assert _C._host is not None
    monkeypatch.setattr(_C, "_host", None)
    monkeypatch.setattr(_C, "_host_failed", True)
    for module in net.modules():
        if hasattr(module, "invalidate_cached_weights"):
            module.invalidate_cached_weights()
    for a, b in zip(with_it, passes()):
        assert torch.equal(a, b)


# (channels, channels, kernel size, stride, transposed, type): one per kernel that addresses rows by 32 bits
@pytest.mark.parametrize("cin,cout,size,stride,transposed,dtype", [
    (128, 128, 3, 1, False, torch.float16), (256, 128, 3, 1, False, torch.bfloat16),
    (128, 256, 2, 2, False, torch.float16), (128, 64, 2, 2, True, torch.float16), (64, 64, 3, 1, False, torch.float16),
    (96, 64, 5, 1, False, torch.float16), (30, 32, 3, 1, False, torch.float16), (64, 64, 1, 1, False, torch.float16),
    (32, 64, 1, 1, False, torch.float32), (32, 32, 1, 2, False, torch.float32), (64, 32, 3, 1, False, torch.float32)])
def test_features_past_the_single_kernel_form(cin, cout, size, stride, transposed, dtype, monkeypatch):
    """Features of 4 GiB and more run as if there were no such form, before and
    after small ones; here from some hundred kilobytes on."""
    gen = torch.Generator(device=DEVICE).manual_seed(cin)
    torch.manual_seed(cin)
    down = minuet.nn.SparseConv3d(4, cin, size, stride=stride, dtype=dtype, device=DEVICE) if transposed else None
    conv = minuet.nn.SparseConv(3, cin, cout, size, stride=stride, transposed=transposed, dtype=dtype, device=DEVICE)
    inputs = []
    for rows in (400, 6000):
        cells = torch.randperm(1 << 15, generator=gen, device=DEVICE)[:rows]
        coordinates = torch.stack([cells >> 10, (cells >> 5) & 31, cells & 31], 1).int()
        coordinates = coordinates[F.build_sorted_index(coordinates)]
        x = minuet.SparseTensor(torch.randn(rows, 4 if transposed else cin, generator=gen, device=DEVICE).to(dtype), coordinates)
        inputs.append(x)

    def results(order):
        cache = minuet.nn.KernelMapCache(3, torch.int32, DEVICE)
        for module in (conv, down) if transposed else (conv,):
            module.set_kernel_map_cache(cache)
            module.invalidate_cached_weights()
            module._routes.clear()
        out = []
        with torch.no_grad():
            for i in order:
                cache.reset()
                x = inputs[i] if down is None else down(inputs[i])
                out.append(conv(x).F)
                assert torch.equal(out[-1], conv(x).F)
        return out

    small, large = results((0, 1))
    calls = []
    for name in ("implicit", "single", "tiled", "pieces"):
        whole = getattr(_C, f"sparse_convolution_forward_{name}")
        monkeypatch.setattr(_C, f"sparse_convolution_forward_{name}",
                            lambda sources, *args, _whole=whole, **kw: calls.append(sources) or _whole(sources, *args, **kw))
    limit = 2000 * cin * dtype.itemsize
    monkeypatch.setattr(_C, "IMPLICIT_MAX_SOURCE_BYTES", limit)
    for got, wanted in zip(results((1, 0, 1, 0, 0, 1)), (large, small, large, small, small, large)):
        # sums of unit normals times uniform weights in another order, rounded once or twice
        tolerance = 1e-5 if dtype == torch.float32 else 4 * torch.finfo(dtype).eps
        assert float((got.double() - wanted.double()).norm() / wanted.double().norm()) < tolerance
    assert calls and all(s.numel() * s.element_size() < limit for s in calls)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("kernel, cin, cout", [(3, 32, 132), (3, 8, 512), (2, 16, 160), (5, 24, 256), (3, 4, 160), (3, 20, 256)])
def test_wide_layers_of_short_rows(kernel, cin, cout, dtype):
    """Past 128 output channels: the single-kernel form, also where rows are padded for it."""
    gen = torch.Generator(device="cuda").manual_seed(cin + cout)
    conv = minuet.nn.SparseConv3d(cin, cout, kernel, dtype=dtype, device="cuda")
    for rows in (1, 700, 10000, 700):
        cells = torch.randperm(1 << 16, generator=gen, device="cuda")[:rows]
        coordinates = torch.stack([cells >> 10, (cells >> 5) & 31, cells & 31], 1).int()
        coordinates = coordinates[minuet.nn.functional.build_sorted_index(coordinates)]
        cache = minuet.nn.KernelMapCache(3, torch.int32, "cuda")
        minuet.set_kernel_map_cache(conv, cache)
        x = minuet.SparseTensor(torch.randn(rows, cin, generator=gen, device="cuda").to(dtype), coordinates)
        with torch.no_grad():
            out = conv(x).F
            assert torch.equal(conv(x).F, out)
        assert len(cache._kernel_maps_cache) == 0
        dense, _ = _C.kernel_map_dense(coordinates, coordinates,
                                       cache._kernel_offsets((1, 1, 1), (kernel,) * 3, (1, 1, 1)), None, None)
        weights = conv.kernel.detach().double()
        wanted, size = (torch.zeros(rows, cout, dtype=torch.float64, device="cuda") for _ in range(2))
        for offset in range(dense.shape[0]):
            hit = (dense[offset] >= 0).nonzero()[:, 0]
            picked = x.F[dense[offset, hit].long()].double()
            wanted[hit] += picked @ weights[offset]
            size[hit] += picked.abs() @ weights[offset].abs()
        # sums of up to 125 x 24 products in 32 bits, one rounding of the result
        assert bool(((out.double() - wanted).abs() <= torch.finfo(dtype).eps * wanted.abs() + 2e-4 * size + 1e-7).all())


@pytest.mark.parametrize("cin, cout, begin", [(64, 256, 100000), (44, 160, 150000), (128, 128, 150000)])
def test_wide_layers_of_many_offsets(cin, cout, begin):
    """5x5x5: the single-kernel form from so many rows on, whichever comes first."""
    gen = torch.Generator(device="cuda").manual_seed(cin)
    torch.manual_seed(cin)
    conv = minuet.nn.SparseConv3d(cin, cout, 5, dtype=torch.float16, device="cuda")
    for rows in (begin, begin - 1, 1000, begin):
        cells = torch.randperm(1 << 21, generator=gen, device="cuda")[:rows]
        coordinates = torch.stack([cells >> 14, (cells >> 7) & 127, cells & 127], 1).int()
        coordinates = coordinates[F.build_sorted_index(coordinates)]
        cache = minuet.nn.KernelMapCache(3, torch.int32, "cuda")
        minuet.set_kernel_map_cache(conv, cache)
        x = minuet.SparseTensor(torch.randn(rows, cin, generator=gen, device="cuda").half(), coordinates)
        with torch.no_grad():
            out = conv(x).F
            dense, _ = _C.kernel_map_dense(coordinates, coordinates, cache._kernel_offsets((1, 1, 1), (5, 5, 5), (1, 1, 1)), None, None)
            pad = -cin % 8
            weights = torch.nn.functional.pad(conv.kernel, (0, 0, 0, pad)).contiguous()
            wanted = _C.sparse_convolution_forward_implicit(torch.nn.functional.pad(x.F, (0, pad)), weights, dense)
            again = conv(x).F
        assert len(cache._kernel_maps_cache) == (rows < begin)
        # (the three kernels round their product rows, of which there are at most 125)
        bound = 125 * 2.0 ** -11 * float(wanted.float().abs().max()) if rows < begin else 0.0
        assert float((out.float() - wanted.float()).abs().max()) <= bound and torch.equal(out, again)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("kernel, cin, cout", [(3, 3, 32), (3, 1, 16), (5, 3, 64), (3, 12, 128), (3, 5, 160), (3, 28, 36)])
def test_padded_layers_from_the_second_call_on(kernel, cin, cout, dtype):
    """Rows that are padded in one launch: the values of the call that pads them step by step, also after the
    weights, the input or the cloud have changed, in a captured graph and from tiles."""
    gen = torch.Generator(device=DEVICE).manual_seed(cin)
    torch.manual_seed(cin)
    conv = minuet.nn.SparseConv3d(cin, cout, kernel, dtype=dtype, device=DEVICE)
    for rows in (1, 333, 20000):
        cells = torch.randperm(1 << 18, generator=gen, device=DEVICE)[:rows]
        coordinates = torch.stack([cells >> 12, (cells >> 6) & 63, cells & 63], 1).int()
        coordinates = coordinates[F.build_sorted_index(coordinates)]
        cache = minuet.nn.KernelMapCache(3, torch.int32, DEVICE)
        minuet.set_kernel_map_cache(conv, cache)
        dense, _ = _C.kernel_map_dense(coordinates, coordinates,
                                       cache._kernel_offsets((1, 1, 1), (kernel,) * 3, (1, 1, 1)), None, None)
        pad = conv._row_padding(torch.empty(0, cin, dtype=dtype, device=DEVICE))
        assert pad > 0
        with torch.no_grad():
            for turn in range(14):
                if turn == 2:
                    conv.kernel.mul_(-0.5)
                features = torch.randn(rows, cin, generator=gen, device=DEVICE).to(dtype)
                got = conv(minuet.SparseTensor(features, coordinates)).F
                wide = torch.nn.functional.pad(features, (0, pad))
                weights = torch.nn.functional.pad(conv.kernel, (0, 0, 0, pad)).contiguous()
                wanted = _C.sparse_convolution_forward_implicit(wide, weights, dense)
                assert turn == 0 or conv._fast is not None
                # (tiles leave out offsets without a source, whose products are zeros)
                assert float((got.float() - wanted.float()).abs().max()) <= 1e-5 * float(wanted.float().abs().max())
            fixed = minuet.SparseTensor(features.clone(), coordinates)
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                out = conv(fixed).F
            for _ in range(3):
                fixed.F.copy_(torch.randn(rows, cin, generator=gen, device=DEVICE))
                graph.replay()
                assert torch.equal(out, conv(fixed).F)


def test_pad_rows_refuses_what_it_cannot_write():
    rows = torch.ones(4, 3, dtype=torch.float16, device=DEVICE)
    out = torch.empty(4, 8, dtype=torch.float16, device=DEVICE)
    call = _C.load_library().mnt_pad_rows
    for arguments in ((rows.data_ptr(), 4, 3, 2, 1, out.data_ptr()), (rows.data_ptr(), 4, 3, 6, 1, out.data_ptr()),
                      (rows.data_ptr(), 4, 3, 8, 0, out.data_ptr()), (rows.data_ptr(), -1, 3, 8, 1, out.data_ptr()),
                      (rows.data_ptr(), 4, 3, 8, 1, out.data_ptr() + 2), (None, 4, 3, 8, 1, out.data_ptr()),
                      (rows.data_ptr(), 1 << 40, 3, 8, 1, out.data_ptr())):
        assert call(*arguments, None) != 0


@pytest.mark.parametrize("dtype, cin, cout, rows, tables", [
    (torch.float32, 3, 64, 1000, 1), (torch.float32, 3, 64, 40000, 0), (torch.float16, 4, 160, 1000, 1),
    (torch.float16, 20, 256, 9000, 0), (torch.float16, 16, 160, 1000, 0), (torch.float32, 4, 64, 1000, 0)])
def test_layers_that_record_gradients_pad_where_it_pays(dtype, cin, cout, rows, tables):
    """The same values with and without a record, whichever form each takes, in both orders."""
    conv, x = layer_and_input(rows, cin, cout, dtype)
    bound = 4 * torch.finfo(dtype).eps if dtype != torch.float32 else 1e-5
    for order in ((True, False), (False, True)):
        results = []
        for recorded in order:
            cache = minuet.nn.KernelMapCache(3, torch.int32, DEVICE)
            minuet.set_kernel_map_cache(conv, cache)
            with torch.set_grad_enabled(recorded):
                for _ in range(2):
                    results.append(conv(x).F.float())
            assert len(cache._kernel_maps_cache) == (tables if recorded else 0)
        for other in results[1:]:
            assert float((other - results[0]).abs().max()) <= bound * 27 * float(results[0].abs().max())


@pytest.mark.parametrize("kind, dtype, kernel, cin, cout, tables", [
    ("plain", torch.float16, 5, 32, 160, {700: 0, 11000: 1, 100000: 0}), ("strided", torch.float16, 5, 64, 160, {150000: 1}),
    ("strided", torch.float16, 5, 32, 160, {11000: 1, 100000: 0}), ("dilated", torch.float16, 5, 128, 128, {150000: 1}),
    ("plain", torch.float32, 4, 16, 80, {700: 0, 50000: 1, 250000: 0}), ("strided", torch.float32, 3, 32, 64, {260000: 1}),
    ("dilated", torch.float32, 3, 16, 96, {50000: 0})])
def test_rules_follow_the_form_of_a_layer(kind, dtype, kernel, cin, cout, tables):
    """What a layer runs on each side of the lines, and that it is the values of the forced three kernels."""
    gen = torch.Generator(device=DEVICE).manual_seed(cin + kernel)
    torch.manual_seed(2)
    conv = minuet.nn.SparseConv3d(cin, cout, kernel, stride=2 if kind == "strided" else 1,
                                  dilation=2 if kind == "dilated" else 1, dtype=dtype, device=DEVICE)
    for turn in range(2):
        for rows, built in tables.items():
            cells = torch.randperm(1 << 21, generator=gen, device=DEVICE)[:rows]
            coordinates = torch.stack([cells >> 14, (cells >> 7) & 127, cells & 127], 1).int()
            coordinates = coordinates[F.build_sorted_index(coordinates)]
            x = minuet.SparseTensor(torch.randn(rows, cin, generator=gen, device=DEVICE).to(dtype), coordinates)
            results = []
            for flow in ("auto", "gather_gemm_scatter"):
                conv._tunable_config["dataflow"] = flow
                cache = minuet.nn.KernelMapCache(3, torch.int32, DEVICE)
                minuet.set_kernel_map_cache(conv, cache)
                with torch.no_grad():
                    results.append(conv(x).F.double())
                    assert torch.equal(conv(x).F.double(), results[-1])
                assert len(cache._kernel_maps_cache) == (built if flow == "auto" else 1)
            # fp16: product rows and both results are rounded to nearest, in the 2-norm 3 x 2^-11 / sqrt(3) = 8.5e-4;
            # fp32: two orders of 27 x 64 additions at most, each about sqrt(27 x 64) x 2^-24 / sqrt(3) = 1.4e-6
            bound = {torch.float32: 3e-6, torch.float16: 1e-3}[dtype]
            assert float((results[0] - results[1]).norm() / results[1].norm()) <= bound

"""1x1x1 layers where more than the values of their operands counts: what torch.mm
gives them has to come out, at the first call and past Python."""
import pytest
import torch
import torch.autograd.forward_ad as forward_ad
from torch.utils._python_dispatch import TorchDispatchMode

import minuet_amd as minuet
from minuet_amd.nn import functional as F

pytestmark = pytest.mark.gpu
DEVICE = torch.device("cuda:0")
ROWS = 600
# wider than the kernel for one offset takes, either way; in pieces and narrow; 16 bits
SHAPES = [(256, 128, torch.float32), (64, 256, torch.float32), (64, 32, torch.float32), (16, 32, torch.float32),
          (64, 64, torch.float16)]


def layer(cin, cout, dtype, kept=True, bias=False):
    torch.manual_seed(cin + cout)
    conv = minuet.nn.SparseConv3d(cin, cout, 1, bias=bias, dtype=dtype, device=DEVICE).requires_grad_(False)
    coordinates = torch.zeros(ROWS, 3, dtype=torch.int32, device=DEVICE)
    coordinates[:, 2] = torch.arange(ROWS, device=DEVICE)
    x = torch.randn(ROWS, cin, device=DEVICE).to(dtype)
    call = lambda features, **options: conv(minuet.SparseTensor(features, coordinates), **options).F
    if kept:
        call(x)
        call(x)                                          # (the extension module has its Layer)
    return conv, x, call


def bound(dtype):
    return dict(rtol=2e-3, atol=2e-3) if dtype == torch.float16 else dict(rtol=0, atol=1e-5)


@pytest.mark.parametrize("kept", [False, True])
@pytest.mark.parametrize("cin, cout, dtype", SHAPES)
def test_tangents(cin, cout, dtype, kept):
    conv, x, call = layer(cin, cout, dtype, kept)
    w = conv.kernel[0]
    dx, dw, residual = torch.randn_like(x), torch.randn_like(conv.kernel), torch.randn(ROWS, cout, device=DEVICE).to(dtype)
    for _ in range(2):
        with forward_ad.dual_level():
            out = forward_ad.unpack_dual(call(forward_ad.make_dual(x, dx)))
            assert torch.allclose(out.primal, x @ w, **bound(dtype)) and torch.allclose(out.tangent, dx @ w, **bound(dtype))
            out = forward_ad.unpack_dual(call(x, epilogue=F.Epilogue(residual=forward_ad.make_dual(residual, residual))))
            assert out.tangent is not None and torch.equal(out.tangent, residual)
        tangent = torch.func.jvp(
            lambda k: torch.func.functional_call(conv, {"kernel": k}, (minuet.SparseTensor(x, x[:, :3].int()),)).F,
            (conv.kernel.detach(),), (dw,))[1]
        assert torch.allclose(tangent, x @ dw[0], rtol=1e-2, atol=0.1 if dtype == torch.float16 else 1e-3)


@pytest.mark.parametrize("kept", [False, True])
@pytest.mark.parametrize("cin, cout, dtype", SHAPES)
def test_gradient_of_a_residual(cin, cout, dtype, kept):
    """The layer's own parameters and input record none."""
    conv, x, call = layer(cin, cout, dtype, kept)
    residual = torch.randn(ROWS, cout, device=DEVICE).to(dtype).requires_grad_()
    call(x, epilogue=F.Epilogue(residual=residual)).sum().backward()
    assert torch.equal(residual.grad, torch.ones_like(residual))


@pytest.mark.parametrize("kept", [False, True])
@pytest.mark.parametrize("cin, cout, dtype", SHAPES)
def test_vmap_and_trace(cin, cout, dtype, kept):
    conv, x, call = layer(cin, cout, dtype, kept)
    several = torch.stack([x, -x, x + 1])
    assert torch.allclose(torch.vmap(call)(several), several @ conv.kernel[0], **bound(dtype))
    traced = torch.jit.trace(call, (x,), check_trace=False)
    assert torch.allclose(traced(x + 1), (x + 1) @ conv.kernel[0], **bound(dtype))


class Seen(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.names = []

    def __torch_dispatch__(self, function, types, args=(), kwargs=None):
        self.names.append(function)
        return function(*args, **(kwargs or {}))


@pytest.mark.parametrize("kept", [False, True])
@pytest.mark.parametrize("cin, cout, dtype", SHAPES)
def test_dispatch_modes_and_autocast(cin, cout, dtype, kept):
    conv, x, call = layer(cin, cout, dtype, kept)
    with Seen() as seen:
        call(x)
    assert torch.ops.aten.mm.default in seen.names
    # layers that one kernel has always taken have nothing to do with autocast
    wide = cin * dtype.itemsize > 512 or cout > 128
    for _ in range(2):
        with torch.autocast("cuda", dtype=torch.bfloat16):
            assert call(x).dtype == (torch.bfloat16 if wide else dtype)
        assert call(x).dtype == dtype


@pytest.mark.parametrize("size", [1, 3])
@pytest.mark.parametrize("cin, cout, dtype", SHAPES)
def test_parameters_made_in_inference_mode(cin, cout, dtype, size):
    """They count no versions, so that nothing derived from them can be kept."""
    with torch.inference_mode():
        conv = minuet.nn.SparseConv3d(cin, cout, size, dtype=dtype, device=DEVICE)
        conv.set_kernel_map_cache(minuet.nn.KernelMapCache(3, torch.int32, DEVICE))
        cells = torch.randperm(4096, device=DEVICE)[:ROWS]
        coordinates = torch.stack([cells >> 8, (cells >> 4) & 15, cells & 15], 1).int()
        coordinates = coordinates[F.build_sorted_index(coordinates)]
        x = minuet.SparseTensor(torch.randn(ROWS, cin, device=DEVICE).to(dtype), coordinates)
        first = conv(x).F.clone()
        assert conv(x).F.equal(first)
        conv.kernel.mul_(2.0)
        # (twice the sums, rounded: a result below the normal numbers may be off by their spacing)
        spacing = 2.0 ** -24 if dtype == torch.float16 else 0.0
        for _ in range(2):
            assert ((conv(x).F.double() - 2 * first.double()).abs() <= spacing).all()

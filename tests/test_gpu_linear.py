"""A classifier's head by the kernel that is a wavefront per output."""
import pytest
import torch
from torch import nn

from minuet_amd.nn.functional import _C
from minuet_amd.resnet import _classify

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows,channels,classes,shift", [(1, 1, 1, 0), (3, 63, 5, 0), (8, 256, 10, 0), (2, 520, 3, 4),
                                                         (5, 66, 7, 0), (4, 1032, 13, 1)])
def test_linear_is_the_layer(dtype, rows, channels, classes, shift):
    torch.manual_seed(channels)
    head = nn.Linear(channels, classes, dtype=dtype, device="cuda").requires_grad_(False)
    x = torch.randn(rows * channels + shift, device="cuda").to(dtype)[shift:].view(rows, channels)
    got = _classify(head, x)
    w, b = head.weight.double(), head.bias.double()
    ref = x.double() @ w.t() + b
    # Sums of `channels` fp32 terms, then one rounding to the type.
    bound = (channels + 2) * 2.0 ** -24 * (x.double().abs() @ w.abs().t() + b.abs()) + torch.finfo(dtype).eps * ref.abs()
    assert got.dtype == dtype and bool(((got.double() - ref).abs() <= bound).all())
    assert torch.equal(_C.linear(x, head.weight, None).double(), _C.linear(x, head.weight, torch.zeros_like(head.bias)).double())


def test_a_watched_head_is_called():
    head = nn.Linear(8, 3, device="cuda").requires_grad_(False)
    seen = []
    head.register_forward_hook(lambda *_: seen.append(1))
    _classify(head, torch.ones(2, 8, device="cuda"))
    assert seen == [1]
    learns = nn.Linear(8, 3, device="cuda")
    assert _classify(learns, torch.ones(2, 8, device="cuda")).requires_grad

"""Layer calls from the second on, which take the extension module's way."""
import pytest
import torch

import minuet_amd as minuet
from minuet_amd.nn import functional as F

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

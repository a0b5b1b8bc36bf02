"""16-bit transposed layers whose kernel is their stride: one source a target."""
import pytest
import torch

import minuet_amd as minuet
from minuet_amd.nn import functional as F
from minuet_amd.nn.functional import _C

pytestmark = pytest.mark.gpu


def _map(targets, sources, gen, empty=0.1, double=0.0):
    dense = torch.full((8, targets), -1, dtype=torch.int32)
    offset = torch.randint(0, 8, (targets,), generator=gen)
    source = torch.randint(0, sources, (targets,), generator=gen, dtype=torch.int32)
    source[torch.rand(targets, generator=gen) < empty] = -1
    dense[offset, torch.arange(targets)] = source
    twice = torch.rand(targets, generator=gen) < double
    dense[(offset + 3) % 8, torch.arange(targets)] = torch.where(twice, source, -1).int()
    return dense


def _oracle(dense, x, w):
    out = torch.zeros(dense.shape[1], w.shape[2], dtype=torch.float64)
    for o in range(8):
        t = torch.nonzero(dense[o] >= 0)[:, 0]
        out[t] += x[dense[o][t].long()].double() @ w[o].double()
    return out


# workgroups of 128 targets, of one that is not full, of a share of the chip in one round and in several
@pytest.mark.parametrize("targets", [1, 127, 129, 5000, 60000, 90001, 300007])
@pytest.mark.parametrize("K, N, dtype", [(72, 8, torch.float16), (128, 64, torch.float16), (136, 40, torch.bfloat16),
                                         (256, 128, torch.bfloat16), (200, 72, torch.float16), (160, 144, torch.float16)])
@pytest.mark.parametrize("double", [0.0, 0.001])
def test_one_source_a_target(targets, K, N, dtype, double):
    """(Targets with two sources are not what the kernel is for, and right all the same.)"""
    gen = torch.Generator().manual_seed(targets + K)
    sources = targets // 3 + 2
    dense = _map(targets, sources, gen, double=double)
    x = torch.randn(sources, K, generator=gen).to(dtype)
    w = (torch.randn(8, K, N, generator=gen) / K ** 0.5).to(dtype)
    got = _C.sparse_convolution_forward_single(x.cuda(), w.cuda(), dense.cuda(), F.pack_weights(w.cuda())).cpu()
    expected = _oracle(dense, x, w)
    # fp32 sums of up to 2 K products, rounded once; sums of unit normals over sqrt(K) stay below 8
    bound = expected.abs() * torch.finfo(dtype).eps + 8 * 2.0 ** -24 * (2 * K) ** 0.5
    assert bool(((got.double() - expected).abs() <= bound).all())


def test_epilogue_and_weights_that_are_not_finite():
    gen = torch.Generator().manual_seed(3)
    dense = _map(700, 300, gen)
    x, w = torch.randn(300, 96, generator=gen).half(), (torch.randn(8, 96, 48, generator=gen) / 10).half()
    epilogue = _C.Epilogue(torch.rand(48).cuda(), torch.randn(48).cuda(), torch.randn(700, 48).half().cuda(), "relu")
    x, dense, w = x.cuda(), dense.cuda(), w.cuda()
    other = _C.sparse_convolution_forward_implicit(x, w, dense, epilogue=epilogue)
    w[5, 3, 7] = float("inf")
    got = _C.sparse_convolution_forward_single(x, w, dense, F.pack_weights(w), epilogue=epilogue)
    hit = torch.zeros(700, 48, dtype=torch.bool, device="cuda")
    hit[dense[5] >= 0, 7] = True                 # what uses that weight, and nothing else, is not finite
    assert bool(got[~hit].isfinite().all()) and torch.allclose(got[~hit], other[~hit], rtol=2e-3, atol=2e-3)


# the last of many workgroups and the only one; each wavefront's offset, those that list targets without a
# source among them; maps that keep the promise and one that does not
@pytest.mark.parametrize("targets", [20, 700, 40000])
@pytest.mark.parametrize("double", [0.0, 0.02])
def test_weights_that_are_not_finite_reach_their_targets_only(targets, double):
    gen = torch.Generator().manual_seed(targets)
    dense = _map(targets, 300, gen, empty=0.3, double=double)
    dense[:, targets // 2:targets // 2 + 8] = -1
    x, w = torch.randn(300, 136, generator=gen).half().cuda(), (torch.randn(8, 136, 48, generator=gen) / 12).half().cuda()
    dense = dense.cuda()
    plain = _C.sparse_convolution_forward_single(x, w, dense, F.pack_weights(w))
    assert bool(plain.isfinite().all()) and bool((plain[(dense < 0).all(0)] == 0).all())
    for offset in range(8):
        spoilt = w.clone()
        spoilt[offset, 130, 7], spoilt[offset, 0, 40] = float("inf"), float("nan")
        got = _C.sparse_convolution_forward_single(x, spoilt, dense, F.pack_weights(spoilt))
        reached = torch.zeros(targets, 48, dtype=torch.bool, device="cuda")
        reached[:, [7, 40]] = (dense[offset] >= 0)[:, None]
        assert torch.equal(got[~reached], plain[~reached]) and not bool(got[reached].isfinite().any())


def test_layer_takes_it():
    """Down and up again, through the first call, the second and a planned pass."""
    gen = torch.Generator().manual_seed(1)
    coordinates = torch.unique(torch.randint(0, 24, (5000, 3), generator=gen, dtype=torch.int32), dim=0).cuda()
    coordinates = coordinates[F.build_sorted_index(coordinates)]
    down = minuet.nn.SparseConv3d(32, 128, 2, stride=2, dtype=torch.float16, device="cuda")
    up = minuet.nn.SparseConv(3, 128, 64, 2, stride=2, transposed=True, dtype=torch.float16, device="cuda")
    net = torch.nn.Sequential(down, up)
    cache = minuet.nn.KernelMapCache(ndim=3, dtype=torch.int32, device="cuda")
    minuet.set_kernel_map_cache(net, cache)
    x = minuet.SparseTensor(torch.randn(len(coordinates), 32, generator=gen).half().cuda(), coordinates)
    with torch.no_grad():
        first = net(x).F.clone()
        assert up._has_single_sources(torch.empty(1, 128, dtype=torch.float16, device="cuda"))
        for _ in range(3):
            assert net(x).F.equal(first)
            cache.reset()
        minuet.set_kernel_map_cache(net, minuet.nn.KernelMapCache(ndim=3, dtype=torch.int32, device="cuda"))
        up.tunable_config["dataflow"] = "gather_gemm_scatter"
        other = net(x).F
    assert torch.allclose(first, other, rtol=4e-3, atol=4e-3)

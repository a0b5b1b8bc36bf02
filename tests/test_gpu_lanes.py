"""fp32 layers that multiply hits only, with weights as given and in lane order:
every workgroup shape, channel counts that fill no block, targets that fill no
workgroup."""
import pytest
import torch

import minuet_amd as minuet
from minuet_amd.nn import functional as F
from minuet_amd.nn.functional import _C

pytestmark = pytest.mark.gpu


def _case(targets, offsets, K, N, density, seed):
    gen = torch.Generator().manual_seed(seed)
    sources = targets + 3
    dense = torch.randint(0, sources, (offsets, targets), generator=gen, dtype=torch.int32)
    dense[torch.rand(offsets, targets, generator=gen) >= density] = -1
    x = torch.randn(sources, K, generator=gen)
    w = torch.randn(offsets, K, N, generator=gen) / (K * offsets * density) ** 0.5
    return dense, x, w


def _oracle(dense, x, w):
    out = torch.zeros(dense.shape[1], w.shape[2], dtype=torch.float64)
    for o in range(dense.shape[0]):
        t = torch.nonzero(dense[o] >= 0)[:, 0]
        out[t] += x[dense[o][t].long()].double() @ w[o].double()
    return out


# workgroups of 64 targets and 16 channels to a compute unit pick the shape: from a handful to several
@pytest.mark.parametrize("targets", [1, 15, 17, 130, 700, 2100, 5003, 9001, 20011])
@pytest.mark.parametrize("offsets, K, N", [(27, 32, 32), (8, 64, 128), (27, 20, 36), (2, 4, 4), (27, 80, 64)])
def test_lane_order_is_the_same_product(targets, offsets, K, N):
    dense, x, w = _case(targets, offsets, K, N, 0.3, targets + K)
    expected = _oracle(dense, x, w)
    dense, x, w = dense.cuda(), x.cuda(), w.cuda()
    plain = _C.sparse_convolution_forward_implicit(x, w, dense)
    lanes = _C.sparse_convolution_forward_implicit(x, w, dense, packed_weights=_C.pack_weights_in_lanes(w))
    # fp32 sums of up to offsets * K products of two unit normals over sqrt(their number)
    bound = 8 * 2.0 ** -24 * (offsets * K) ** 0.5
    assert (plain.cpu().double() - expected).abs().max() < bound
    assert lanes.equal(plain)


# 0.9, 1, 1.9, 2, 2.25, 2.3, 2.9, 3, 4.7 and 4.8 workgroups of 64 targets and 16 channels to each of 256 compute units:
# both sides of every line of the layers with one step of 16 channels, with one and a half, and of [O][K][N] ones
@pytest.mark.parametrize("targets", [3790, 4100, 7800, 8200, 9150, 9300, 11900, 12300, 19300, 19700])
@pytest.mark.parametrize("offsets, K, N", [(27, 8, 64), (8, 16, 64), (27, 24, 64), (27, 32, 64), (2, 80, 64)])
def test_lane_order_at_the_lines_between_shapes(targets, offsets, K, N):
    dense, x, w = _case(targets, offsets, K, N, 0.2, targets + K)
    expected = _oracle(dense, x, w)
    dense, x, w = dense.cuda(), x.cuda(), w.cuda()
    plain = _C.sparse_convolution_forward_implicit(x, w, dense)
    lanes = _C.sparse_convolution_forward_implicit(x, w, dense, packed_weights=_C.pack_weights_in_lanes(w))
    # as above; the density is of the whole map, single targets have up to all offsets
    assert (plain.cpu().double() - expected).abs().max() < 8 * 2.0 ** -24 * (offsets * K / 0.2) ** 0.5
    assert lanes.equal(plain)


@pytest.mark.parametrize("activation", [None, "relu"])
def test_lane_order_epilogue(activation):
    dense, x, w = (t.cuda() for t in _case(333, 27, 48, 72, 0.4, 5))
    epilogue = _C.Epilogue(torch.rand(72).cuda(), torch.randn(72).cuda(), torch.randn(333, 72).cuda(), activation)
    plain = _C.sparse_convolution_forward_implicit(x, w, dense, epilogue=epilogue)
    lanes = _C.sparse_convolution_forward_implicit(x, w, dense, epilogue=epilogue,
                                                   packed_weights=_C.pack_weights_in_lanes(w))
    assert lanes.equal(plain)


def test_lane_weights_follow_the_parameter():
    coordinates = torch.unique(torch.randint(0, 12, (900, 3), generator=torch.Generator().manual_seed(1),
                                             dtype=torch.int32), dim=0).cuda()
    coordinates = coordinates[F.build_sorted_index(coordinates)]
    conv = minuet.nn.SparseConv3d(32, 32, 3, device="cuda")
    conv.set_kernel_map_cache(minuet.nn.KernelMapCache(ndim=3, dtype=torch.int32, device="cuda"))
    x = minuet.SparseTensor(torch.randn(len(coordinates), 32, device="cuda"), coordinates)
    with torch.no_grad():
        first = conv(x).F.clone()
        assert conv(x).F.equal(first)                                  # (and past Python)
        conv.kernel.mul_(2.0)                                          # in place: same storage, new version
        assert conv(x).F.equal(2 * first)
        assert conv(x).F.equal(2 * first)
    assert conv(x).F.detach().equal(2 * first)                         # gradients are recorded: as they are


# hits only, of three kinds of map; the channels in pieces, wider than the library's product was left for either way
@pytest.mark.parametrize("cin, cout, size, stride, transposed", [
    (32, 32, 3, 1, False), (64, 128, 2, 2, False), (64, 32, 2, 2, True), (256, 128, 1, 1, False), (64, 256, 1, 1, False)])
def test_layers_read_the_parameter_itself(cin, cout, size, stride, transposed):
    """A write through ``.data`` leaves no mark on the parameter, one of the caller's
    before a replay none that a captured pass could see."""
    coordinates = torch.unique(torch.randint(0, 12, (900, 3), generator=torch.Generator().manual_seed(1),
                                             dtype=torch.int32), dim=0).cuda()
    coordinates = coordinates[F.build_sorted_index(coordinates)]
    cache = minuet.nn.KernelMapCache(ndim=3, dtype=torch.int32, device="cuda")
    conv = minuet.nn.SparseConv(3, cin, cout, size, stride=stride, transposed=transposed, device="cuda")
    conv.set_kernel_map_cache(cache)
    x = minuet.SparseTensor(torch.randn(len(coordinates), cin, device="cuda"), coordinates)
    with torch.no_grad():
        if transposed:
            down = minuet.nn.SparseConv3d(cin, cin, size, stride=stride, device="cuda")
            down.set_kernel_map_cache(cache)
            x = down(x)
        first = conv(x).F.clone()
        assert conv(x).F.equal(first)                                  # (and past Python)
        conv.kernel.mul_(2.0)                                          # in place: same storage, new version
        assert conv(x).F.equal(2 * first)
        assert conv(x).F.equal(2 * first)
        conv.kernel.data.mul_(2.0)                                     # same storage, same version
        assert conv(x).F.equal(4 * first)
        conv._fast = None
        conv.kernel.data.mul_(2.0)
        assert conv(x).F.equal(8 * first)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = conv(x).F
        for _ in range(3):
            conv.kernel.mul_(0.5)
            out.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert out.equal(conv(x).F)
        assert out.equal(first)
    assert conv(x).F.detach().allclose(first, rtol=0, atol=2e-5)       # gradients are recorded: as they are


def test_refuses_another_layer_s_weights():
    dense, x, w = (t.cuda() for t in _case(50, 27, 32, 32, 0.3, 2))
    with pytest.raises((RuntimeError, ValueError)):
        _C.sparse_convolution_forward_implicit(x, w, dense, packed_weights=_C.pack_weights_in_lanes(w[:8]))
    with pytest.raises((RuntimeError, ValueError)):
        _C.sparse_convolution_forward_implicit(x[:, :32].half(), w.half(), dense,
                                               packed_weights=_C.pack_weights_in_lanes(w))


# one workgroup and several, rows that fill none, pieces of 16 and of 32 channels, channels that fill no block
@pytest.mark.parametrize("rows", [1, 33, 700, 5003])
@pytest.mark.parametrize("K, N", [(48, 32), (64, 64), (128, 20), (256, 128), (512, 36)])
def test_pointwise_layer_in_pieces(rows, K, N):
    gen = torch.Generator().manual_seed(rows + K)
    x, w = torch.randn(rows, K, generator=gen), torch.randn(K, N, generator=gen) / K ** 0.5
    residual = torch.randn(rows, N, generator=gen)
    pieces = F.channel_pieces(K)
    packed = _C.pack_weights_in_lanes(w.view(pieces, K // pieces, N).cuda())
    got = _C.sparse_convolution_forward_pieces(x.cuda(), packed, N, _C.Epilogue(residual=residual.cuda())).cpu()
    plain = w.view(pieces, K // pieces, N).cuda()
    assert got.cuda().equal(_C.sparse_convolution_forward_pieces(x.cuda(), plain, N, _C.Epilogue(residual=residual.cuda())))
    expected = x.double() @ w.double() + residual.double()
    assert (got.double() - expected).abs().max() < 8 * 2.0 ** -24 * K ** 0.5
    with pytest.raises((RuntimeError, ValueError)):
        _C.sparse_convolution_forward_pieces(x.cuda(), packed, N + 16)
    with pytest.raises((RuntimeError, ValueError)):
        _C.sparse_convolution_forward_pieces(x.cuda(), plain, N + 4)


def test_pointwise_layer_takes_pieces_by_its_rows():
    conv = minuet.nn.SparseConv3d(128, 64, 1, bias=True, device="cuda")
    most = F.pieces_rows_limit(128, 64, torch.float32)
    x = torch.randn(most + 5, 128, device="cuda")
    coordinates = torch.zeros(most + 5, 3, dtype=torch.int32, device="cuda")
    coordinates[:, 2] = torch.arange(most + 5)
    with torch.no_grad():
        expected = (x.double() @ conv.kernel[0].double() + conv.bias.double()).float()
        for rows in (900, 900, most, most + 1, most + 5, 37, most + 1):
            out = conv(minuet.SparseTensor(x[:rows], coordinates[:rows]))
            assert torch.allclose(out.F, expected[:rows], rtol=0, atol=2e-5)
        conv.kernel.mul_(2.0)
        out = conv(minuet.SparseTensor(x[:900], coordinates[:900]))
        assert torch.allclose(out.F, 2 * expected[:900] - conv.bias, rtol=0, atol=4e-5)

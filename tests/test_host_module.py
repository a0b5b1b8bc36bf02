"""The extension module with the host side of layer calls, as far as it needs no GPU."""
import warnings

import pytest
import torch
import torch.nn.utils.prune

import minuet_amd as minuet
from minuet_amd.nn.functional import _C


def test_what_torch_throws_reaches_the_caller():
    """A tensor without storage (here a sparse one) makes const_data_ptr throw
    inside the module: a Python exception, not the end of the process."""
    host = _C.load_host()
    norm = minuet.nn.BatchNorm(4).eval()
    norm._buffers["running_mean"] = torch.zeros(4).to_sparse()
    with pytest.raises(RuntimeError):
        host.Affine(norm, torch.ones(4), torch.zeros(4))
    conv = minuet.nn.SparseConv3d(4, 4, 3)
    weights, conv._parameters["kernel"] = conv.kernel.detach(), conv.kernel.detach().to_sparse()
    with pytest.raises(RuntimeError):
        host.Layer(conv, host.IMPLICIT, weights, weights, None, 0)
    conv._parameters["kernel"] = weights                 # and the module is as usable as before
    assert type(host.Layer(conv, host.IMPLICIT, weights, weights, None, 0)) is host.Layer


@pytest.mark.parametrize("name", ["kernel", "bias"])
def test_no_layer_for_parameters_made_from_others(name):
    host = _C.load_host()
    conv = minuet.nn.SparseConv3d(4, 4, 3, bias=True)
    torch.nn.utils.prune.identity(conv, name)
    weights = conv.kernel.detach()
    with pytest.raises(ValueError, match="its own parameters"):
        host.Layer(conv, host.IMPLICIT, weights, weights, None, 0)


def test_library_does_without_the_module(monkeypatch, tmp_path):
    """Where it can be neither loaded nor built, one warning and None."""
    from minuet_amd import build

    def no_compiler():
        raise RuntimeError("no compiler here")
    monkeypatch.setattr(_C, "_host", None)
    monkeypatch.setattr(_C, "_host_failed", False)
    monkeypatch.setattr(build, "HOST_PATH", str(tmp_path / "minuet_host.so"))
    monkeypatch.setattr(build, "build_host", no_compiler)
    with pytest.warns(RuntimeWarning, match="no compiler here"):
        assert _C.load_host() is None
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert _C.load_host() is None


def test_no_thread_local_data_in_the_module():
    """Thread-local data that nothing reads, in a module loaded late, makes glibc
    before 2.39 take the slow way to that of every library: 20 % on the host side
    of each torch operation (ELF program headers of type 7 say that there is some)."""
    import struct
    from minuet_amd.build import HOST_PATH
    _C.load_host()
    with open(HOST_PATH, "rb") as f:
        header = f.read(64)
        assert header[:6] == b"\x7fELF\x02\x01"
        at, (size, count) = struct.unpack_from("<Q", header, 32)[0], struct.unpack_from("<HH", header, 54)
        f.seek(at)
        kinds = [struct.unpack_from("<I", f.read(size))[0] for _ in range(count)]
    assert 7 not in kinds
